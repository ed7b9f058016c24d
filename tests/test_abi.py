"""The C-ABI library loads and exports every symbol the header declares
(no compute calls: this runs without a GPU)."""

import ctypes
import os
import re

import pytest

from veloxquant_mlx_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "veloxquant_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vq_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    assert _declared() == sorted(_lib.EXPORTED_SYMBOLS)


def test_library_exports_every_declared_symbol():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail(f"{_lib.LIB_PATH} is missing: run `python -m veloxquant_mlx_amd.build`")
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in _declared():
        assert hasattr(lib, name), name
    assert lib.vq_abi_version() == 16


def test_attend_args_struct_matches_header_field_order():
    text = open(os.path.join(ROOT, "include", "veloxquant_hip.h")).read()
    body = text[text.index("typedef struct vq_attend_args {"):text.index("} vq_attend_args;")]
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    names = []
    for decl in body.split(";"):
        decl = decl.split("{")[-1].strip()
        if not decl:
            continue
        for part in decl.split(","):
            names.append(re.findall(r"[A-Za-z_][A-Za-z0-9_]*", part)[-1])
    assert names == [f[0] for f in _lib.AttendArgs._fields_]


def test_argument_errors_surface_without_a_gpu():
    lib = _lib.load()
    # invalid axis is rejected before any device work
    rc = lib.vq_kivi_quant_dequant(None, None, 0, 1, 4, 8, 7, 32, 3, 1e-8, None)
    assert rc == _lib.VQ_ERR_INVALID
    assert "axis must be -1 or -2" in _lib.last_error()
    with pytest.raises(ValueError, match="axis must be -1 or -2"):
        _lib.check(rc)
    a = _lib.AttendArgs()
    a.B, a.Hq, a.Hkv, a.Sq, a.D = 1, 6, 4, 1, 128
    a.n_tail = 4
    assert lib.vq_kivi_attend(a) == _lib.VQ_ERR_INVALID
    assert "multiple of H_kv" in _lib.last_error()
    # ready-made tiles: a missing or short buffer is refused by the writer and by the attention call
    t = _lib.AttendArgs()
    t.B, t.Hq, t.Hkv, t.Sq, t.D = 1, 4, 4, 1, 128
    t.n_tail = 64
    assert lib.vq_kivi_prefill_tiles(t, 0, 2) == _lib.VQ_ERR_INVALID
    assert "kv_tiles must be given" in _lib.last_error()
    t.kv_tiles, t.tile_cap = 4096, 1
    assert lib.vq_kivi_prefill_tiles(t, 0, 2) == _lib.VQ_ERR_INVALID
    assert "do not lie inside" in _lib.last_error()
    assert lib.vq_kivi_attend(t) == _lib.VQ_ERR_INVALID
    assert "room for all 64 slots" in _lib.last_error()



def test_packed_argument_block_is_the_structure():
    """The decode step's argument block, packed by ``struct``, lands in the fields of the ctypes mirror."""
    values = [0.5 if t is _lib.f32 else i + 1 for i, (_, t) in enumerate(_lib.AttendArgs._fields_)]
    a = _lib.AttendArgs.from_buffer_copy(_lib.ATTEND_PACK.pack(*values))
    assert [getattr(a, n) for n, _ in _lib.AttendArgs._fields_] == values


@pytest.mark.parametrize("lens", [None, "seq_lens", "packed_lens"])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,D,n_packed,n_tail,window,pairs", [
    (1, 64, 8, 1, 128, 32768, 128, 1024, 0), (2, 64, 8, 1, 128, 32768, 128, 4096, 0),      # a window far below the context
    (7, 12, 4, 1, 256, 20000, 140, 1024, 0), (8, 40, 10, 1, 128, 8192, 130, 512, 0),
    (2, 32, 8, 4, 128, 8192, 128, 1024, 0), (2, 12, 4, 4, 128, 8192, 128, 1024, 0),        # several positions; groups filled up
    (2, 14, 2, 16, 64, 4096, 7, 100, 0), (3, 40, 2, 32, 128, 4096, 50, 64, 0),             # vector kernel; groups of more than eight
    (16, 32, 8, 128, 128, 0, 128, 0, 0), (2, 32, 32, 700, 128, 0, 700, 99, 0),             # a right-padded prompt over plain rows
    (3, 32, 4, 1, 128, 8192, 33, 200, 8), (2, 12, 2, 1, 128, 2048, 64, 0, 3)])             # heads of 64 channels in pairs
def test_workspace_query_covers_the_call_that_runs(B, Hq, Hkv, Sq, D, n_packed, n_tail, window, pairs, lens):
    """What the query answers is what the call asks for, with lengths a sequence and without (the call is refused for want of
    any workspace, before a launch)."""
    lib = _lib.load()
    a = _lib.AttendArgs()
    a.B, a.Hq, a.Hkv, a.Sq, a.D, a.n_packed, a.n_tail, a.sliding_window = B, Hq, Hkv, Sq, D, n_packed, n_tail, window
    a.pack_bits, a.group, a.meta_dtype, a.v_layout, a.cap_tokens, a.tail_cap = 4, 32, 0, 1, 32768, 768
    a.q_dtype = a.out_dtype = a.tail_dtype = 0
    a.scale, a.causal = 0.1, int(Sq > 1)
    for f in ("q", "out", "sync_counters") + (("k_packed", "k_scale", "k_zero", "v_packed", "v_scale", "v_zero") if n_packed else ()):
        setattr(a, f, 4096)
    a.k_tail = a.v_tail = 4096
    if lens == "packed_lens":
        a.packed_lens = a.tail_lens = 4096
    x = _lib.AttendExt(pairs, 4096 if lens == "seq_lens" else None) if pairs or lens == "seq_lens" else None
    need = lib.vq_kivi_attend_workspace_ext(a, x)
    assert need == lib.attend_packed_workspace(bytes(a), None if x is None else bytes(x))
    if x is None:
        assert need == lib.vq_kivi_attend_workspace(a)
    if need == 0:
        return   # the launch writes its output itself: nothing refuses the call
    assert lib.vq_kivi_attend_ext(a, x) == _lib.VQ_ERR_WORKSPACE
    assert int(re.search(r"workspace of (\d+) bytes required", _lib.last_error()).group(1)) == need


def test_half_a_pair_of_length_lists_is_refused():
    """packed_lens and tail_lens go together, with the extension and without: one list alone is the library's own form of
    one length a sequence and never a caller's."""
    lib = _lib.load()
    a = _lib.AttendArgs()
    a.B, a.Hq, a.Hkv, a.Sq, a.D, a.n_tail, a.tail_cap, a.scale = 2, 4, 4, 1, 128, 64, 64, 0.1
    a.q = a.out = a.k_tail = a.v_tail = 4096
    for field in ("packed_lens", "tail_lens"):
        setattr(a, field, 4096)
        for x in (None, _lib.AttendExt(0, 4096)):
            assert lib.vq_kivi_attend_ext(a, x) == lib.vq_kivi_attend(a) == _lib.VQ_ERR_INVALID
            assert "go together" in _lib.last_error()
        setattr(a, field, None)
    a.packed_lens = a.tail_lens = 4096
    assert lib.vq_kivi_attend_ext(a, _lib.AttendExt(0, 4096)) == _lib.VQ_ERR_INVALID and "exclude" in _lib.last_error()


@pytest.mark.parametrize("D,Hq,Hkv,B,n_packed,n_tail,splits", [
    (128, 40, 10, 2, 32000, 100, 13), (128, 28, 4, 9, 8192, 150, 7), (128, 32, 8, 6, 4224, 140, 5), (128, 32, 8, 9, 8192, 0, 3),
    (128, 40, 10, 9, 20000, 150, 3), (128, 28, 4, 15, 32768, 129, 4), (128, 8, 1, 50, 4096, 33, 5), (256, 12, 4, 6, 20000, 140, 11),
    (256, 12, 4, 7, 8960, 140, 9), (256, 12, 4, 10, 20000, 0, 7), (256, 8, 4, 10, 20000, 1, 7)])
def test_a_fixed_order_cuts_by_shapes_alone(D, Hq, Hkv, B, n_packed, n_tail, splits):
    """Sequences of different lengths: on demand the blocks cut every sequence by all lengths of the batch, also where another launch
    reads the partials; under a fixed order, asked for by the call or the process, the launch has the splits of the shapes.  The workspace is the larger of the two, whichever order the query or the process names."""
    lib = _lib.load()
    a = _lib.AttendArgs()
    a.B, a.Hq, a.Hkv, a.Sq, a.D, a.n_packed, a.n_tail = B, Hq, Hkv, 1, D, n_packed, n_tail
    a.pack_bits, a.group, a.meta_dtype, a.v_layout, a.cap_tokens, a.tail_cap = 2, 32, 0, 1, 32768, 768
    a.scale = 0.1
    for f in ("q", "out", "k_packed", "k_scale", "k_zero", "v_packed", "v_scale", "v_zero", "k_tail", "v_tail", "packed_lens", "tail_lens",
              "sync_counters"):
        setattr(a, f, 4096)

    def nparts(order, num_splits=0):
        path, n = ctypes.c_int(0), ctypes.c_int(0)
        a.fixed_order, a.num_splits = order, num_splits
        assert lib.vq_kivi_attend_plan(a, ctypes.byref(path), ctypes.byref(n)) == 0 and path.value == 1
        return n.value

    by_shapes = nparts(1, splits)
    evened = nparts(2)
    assert evened > by_shapes   # (a shape that is evened)
    assert nparts(1) == nparts(3) == by_shapes
    for field in ("sync_counters", "sink_k"):   # another launch reads the partials
        was, a.sink_v, a.sink_pos, a.sink_cap = getattr(a, field), 4096, 4096, 1
        setattr(a, field, None if was else 4096)
        assert nparts(2) == evened and nparts(1) == by_shapes
        setattr(a, field, was)
    before = lib.vq_kivi_attend_fixed_order(1)
    try:
        assert nparts(0) == by_shapes and nparts(2) > by_shapes
        sizes = set()
        for a.fixed_order in (0, 1, 2, 3):
            sizes.add(lib.vq_kivi_attend_workspace(a))
        lib.vq_kivi_attend_fixed_order(0)
        sizes.add(lib.vq_kivi_attend_workspace(a))
        assert sizes == {B * Hq * nparts(2) * (D + 2) * 4}
    finally:
        lib.vq_kivi_attend_fixed_order(before)
