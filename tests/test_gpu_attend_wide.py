"""Attention with sixteen channels a lane: byte codes with float32 scale / zero against the one-wave-a-row kernel, and
codebook indices against the composition in float64 (veloxquant_mlx/allocators/vecinfer.py:137-184, 321-335)."""

import math

import pytest
import torch

from tests._gpu import require_gpu
from veloxquant_mlx_amd import kernels as K
from veloxquant_mlx_amd.allocators.vecinfer import walsh_hadamard_matrix

pytestmark = pytest.mark.gpu


def _visible(Sq, n, causal, window, device):
    pos, t = torch.arange(n - Sq, n, device=device)[:, None], torch.arange(n, device=device)[None]
    keep = t <= pos if causal else torch.ones((Sq, n), dtype=torch.bool, device=device)
    return keep & (t > pos - window) if window else keep


# tokens round the units of 16 / 32, the shortest split (128) and one with several units a wave; GQA groups of one tile and of
# two; groups of 32 and more; buffers with room to spare
@pytest.mark.parametrize("B,Hq,Hkv,D,n,group,Sq,causal,window,extra", [
    (1, 8, 2, 64, 1, 32, 1, False, 0, 31), (2, 7, 1, 64, 129, 32, 1, False, 0, 0), (1, 4, 4, 128, 33, 64, 1, False, 0, 63),
    (2, 28, 4, 128, 1037, 32, 1, False, 0, 3), (1, 12, 4, 256, 517, 128, 1, False, 0, 0), (1, 2, 1, 256, 95, 32, 3, True, 0, 0),
    (1, 8, 2, 128, 700, 32, 2, True, 0, 4), (1, 4, 2, 128, 900, 32, 1, False, 77, 0), (3, 16, 1, 128, 4099, 96, 1, False, 0, 0),
    # a last tile of one head; positions of one and of three heads in a tile, the last tile short
    (1, 9, 1, 128, 300, 32, 1, False, 0, 0), (2, 3, 3, 64, 200, 32, 6, True, 50, 0), (1, 3, 1, 128, 260, 32, 2, True, 0, 5),
])
def test_byte_codes_against_the_general_kernel(B, Hq, Hkv, D, n, group, Sq, causal, window, extra):
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(n + D)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    cap, codes = n + extra, lambda: torch.randint(0, 2 ** 31 - 1, (B, Hkv, n + extra, D // 4), generator=gen, device="cuda", dtype=torch.int32)
    ks = r(B, Hkv, -(-cap // group), D).abs() * 0.02
    vs = r(B, Hkv, cap, -(-D // group)).abs() * 0.02
    kw = dict(k_packed=codes(), k_scale=ks, k_zero=-128 * ks + r(*ks.shape), v_packed=codes(), v_scale=vs,
              v_zero=-128 * vs + r(*vs.shape), n_packed=n, bits=8, group_size=group, scale=D ** -0.5, causal=causal,
              sliding_window=window, out_dtype=torch.float32)
    q, wide, general = r(B, Hq, Sq, D), {}, {}
    out = K.kivi_packed_attend(q, _plan_out=wide, **kw)
    ref = K.kivi_packed_attend(q, num_splits=-1, _plan_out=general, **kw)
    assert wide["path"] == 4 and general["path"] == 0
    # both rebuild code * scale + zero in float32 and differ by the order of their sums
    assert float((out - ref).abs().max()) < 5e-5
    # one type, group or layout further is the other kernels'
    other = dict(kw, k_scale=ks.half(), k_zero=kw["k_zero"].half(), v_scale=vs.half(), v_zero=kw["v_zero"].half())
    K.kivi_packed_attend(q, _plan_out=wide, **other)
    assert wide["path"] != 4


@pytest.mark.parametrize("B,Hq,Hkv,D,n,Sq,causal,window,nk,sub,rows,cap", [
    (1, 8, 2, 128, 1, 1, False, 0, 4096, 4, 2, 1), (2, 32, 8, 128, 777, 1, False, 0, 4096, 4, 8, 1024), (1, 7, 1, 64, 129, 2, True, 0, 256, 8, 1, 129),
    (1, 12, 4, 256, 500, 1, False, 0, 256, 8, 0, 512), (1, 28, 4, 128, 2049, 1, False, 100, 1024, 4, 4, 2050), (1, 3, 3, 64, 33, 1, True, 0, 256, 4, 1, 64),
    (1, 4, 2, 128, 4100, 4, True, 33, 300, 8, 2, 4100), (1, 4, 2, 64, 300, 21, True, 0, 4096, 4, 2, 300),
])
@pytest.mark.parametrize("q_dtype", [torch.float32, torch.bfloat16])
def test_indices_against_float64(B, Hq, Hkv, D, n, Sq, causal, window, nk, sub, rows, cap, q_dtype):
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(n + nk)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    idx = lambda m, s: torch.randint(0, m, (B, Hkv, cap, D // s), generator=gen, device="cuda",
                                     dtype=torch.uint8 if m <= 256 else torch.int32)
    q, ki, vi, kcb, vcb = r(B, Hq, Sq, D).to(q_dtype), idx(nk, sub), idx(256, 8), r(nk, sub), r(256, 8)
    smooth = r(rows, D).exp() if rows else None
    H = walsh_hadamard_matrix(D, device="cuda")
    scale = 0.3 / math.sqrt(D)
    out = K.vecinfer_attend_indices(q, ki, kcb, vi, vcb, scale, n_tokens=n, smooth=smooth, H_mat=H, causal=causal, sliding_window=window)
    qt = q.double()
    if rows:
        qt = qt * smooth.double().repeat_interleave(Hq // rows if rows > 1 else Hq, 0)[None, :, None]
    qt = qt @ H.double()
    wide = lambda i, cb: cb.double()[i[:, :, :n].long()].reshape(B, Hkv, n, D).repeat_interleave(Hq // Hkv, 1)
    s = (qt[..., None, :] * wide(ki, kcb)[:, :, None]).sum(-1) * scale
    s = s.masked_fill(~_visible(Sq, n, causal, window, "cuda"), -math.inf)
    p = torch.softmax(s, -1)
    ref = (p[..., None] * wide(vi, vcb)[:, :, None]).sum(-2)
    # float32 throughout: a score of |s| carries |s| 2^-24 per addition (D of them at most) into every probability;
    # bfloat16 rounds the output to 2^-9
    tol = float(s[s > -math.inf].abs().max()) * D * 2.0 ** -24 * 2 + 1e-5
    err = (out.double() - ref).abs()
    assert float((err - ref.abs() * (2.0 ** -8 if q_dtype == torch.bfloat16 else 0)).max()) < tol * float(ref.abs().max())


def test_indices_refused_shapes():
    require_gpu()
    z = lambda *s, dtype=torch.float32: torch.zeros(s, device="cuda", dtype=dtype)
    ki, vi, kcb, vcb = z(1, 2, 64, 32, dtype=torch.int32), z(1, 2, 64, 16, dtype=torch.uint8), z(4096, 4), z(256, 8)
    attend = lambda q, ki=ki, vi=vi, kcb=kcb, vcb=vcb: K.vecinfer_attend_indices(q, ki, kcb, vi, vcb, 0.1, n_tokens=64)
    assert attend(z(1, 4, 1, 128)) is not None
    assert attend(z(1, 4, 128, 128)) is None                                # 256 rows a kv head
    assert attend(z(1, 4, 1, 128, dtype=torch.float64)) is None
    assert attend(z(1, 4, 1, 128), ki=z(1, 2, 64, 64, dtype=torch.int32)[..., ::2]) is None
    assert attend(z(1, 4, 1, 128), ki=z(1, 2, 64, 16, dtype=torch.int32), kcb=z(8192, 8)) is None   # codebook past LDS


def _byte_call(B, Hkv, D, n, gen, group=32, bits=8, meta=torch.float32):
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    words = lambda: torch.randint(0, 2 ** 31 - 1, (B, Hkv, n, -(-D // (32 // bits))), generator=gen, device="cuda", dtype=torch.int32)
    ks, vs = r(B, Hkv, -(-n // group), D).abs() * 0.02, r(B, Hkv, n, -(-D // group)).abs() * 0.02
    half = 2.0 ** (bits - 1)
    return dict(k_packed=words(), k_scale=ks.to(meta), k_zero=(-half * ks).to(meta), v_packed=words(), v_scale=vs.to(meta),
                v_zero=(-half * vs).to(meta), n_packed=n, bits=bits, group_size=group, scale=D ** -0.5)


@pytest.mark.parametrize("bits,group,Hq,Hkv,D,path", [(4, 32, 16, 4, 32, 3), (8, 32, 16, 4, 64, 4), (4, 4, 16, 4, 32, 0)])
def test_a_batch_adds_in_the_order_of_its_parts(bits, group, Hq, Hkv, D, path):
    """Under ``fixed_order`` with the same cut, sequences of a large batch (more than 8192 query rows) give the bits that they
    give in a small one: layers stacked into one call against a call a layer."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(bits + D)
    B = 8192 // Hq + 2
    kw = _byte_call(B, Hkv, D, 4096, gen, group, bits)
    q, plan, one = torch.randn((B, Hq, 1, D), generator=gen, device="cuda"), {}, {}
    out = K.kivi_packed_attend(q, fixed_order=True, num_splits=16, _plan_out=plan, **kw)
    assert plan["path"] == path and plan["nparts"] > 8
    at = slice(3, 5)
    part = {name: t[at].contiguous() if isinstance(t, torch.Tensor) else t for name, t in kw.items()}
    few = K.kivi_packed_attend(q[at], fixed_order=True, num_splits=16, _plan_out=one, **part)
    assert one == plan
    assert torch.equal(out[at], few)


@pytest.mark.parametrize("bits,D", [(8, 64), (4, 32)])
def test_an_infinite_value_of_a_run_that_weighs_nothing(bits, D):
    """Sixteen runs, one of which scores so low that its weight underflows, with an infinite value in it: 0 * inf is not a
    number, as in a softmax over all tokens in float32."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(bits)
    kw = _byte_call(1, 1, D, 4096, gen, bits=bits)
    q = torch.ones((1, 1, 1, D), device="cuda")
    kw["k_zero"][:, :, 32:40] -= 300.0        # tokens 1024 .. 1279: a run of their own
    kw["v_zero"][:, :, 1100, 0] = float("inf")
    plan = {}
    out = K.kivi_packed_attend(q, num_splits=16, _plan_out=plan, **kw)
    assert plan["nparts"] == 16
    assert out[..., :32].isnan().all() and out[..., 32:].isfinite().all()


@pytest.mark.parametrize("B,D,n,asked,path", [(64, 128, 36, 0, 4), (65, 128, 36, 0, 3), (65, 128, 37, 0, 4), (65, 128, 36, 1, 4),
                                              (385, 128, 64, 0, 3), (385, 128, 65, 0, 4), (384, 128, 64, 0, 4), (65, 64, 72, 0, 3), (65, 256, 18, 0, 3)])
def test_many_tiles_over_few_tokens_take_the_smaller_blocks(B, D, n, asked, path):
    """Both sides of the rule, against the one-wave-a-row kernel."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(B + n)
    kw, q, plan = _byte_call(B, 4, D, n, gen), torch.randn((B, 8, 1, D), generator=gen, device="cuda"), {}
    out = K.kivi_packed_attend(q, num_splits=asked, _plan_out=plan, **kw)
    ref = K.kivi_packed_attend(q, num_splits=-1, **kw)
    assert plan["path"] == path
    assert float((out - ref).abs().max()) < 5e-5   # (the order of float32 sums over the same rebuilt rows)


@pytest.mark.parametrize("n,asked", [(4096, 16), (4096, 32), (1000, 64), (65536, 512), (257, 2)])
def test_a_given_cut_is_the_same_on_byte_codes(n, asked):
    """``num_splits`` cuts the tokens alike whichever vector kernel takes them: runs of at least 256 tokens, whole 64s -- and so the
    partials a caller has set memory aside for."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(n)
    kw, q = _byte_call(1, 1, 64, n, gen), torch.randn((1, 4, 1, 64), generator=gen, device="cuda")
    wide, rows = {}, {}
    K.kivi_packed_attend(q, num_splits=asked, _plan_out=wide, **kw)
    half = {name: t.half() if name in ("k_scale", "k_zero", "v_scale", "v_zero") else t for name, t in kw.items()}
    K.kivi_packed_attend(q, num_splits=asked, _plan_out=rows, **half)
    assert wide["path"] == 4 and rows["path"] == 3 and wide["nparts"] == rows["nparts"]


def test_byte_codes_of_any_batch_take_one_path():
    """The kernel of a call does not change with the batch while its grid fits: 36 layers of 16 sequences of 8 heads."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(9)
    kw = _byte_call(36 * 16, 8, 64, 33, gen)
    q, plan, one = torch.randn((36 * 16, 8, 1, 64), generator=gen, device="cuda"), {}, {}
    out = K.kivi_packed_attend(q, fixed_order=True, num_splits=1, _plan_out=plan, **kw)
    part = {name: t[:2].contiguous() if isinstance(t, torch.Tensor) else t for name, t in kw.items()}
    few = K.kivi_packed_attend(q[:2], fixed_order=True, num_splits=1, _plan_out=one, **part)
    assert plan["path"] == one["path"] == 4 and torch.equal(out[:2], few)


def test_indices_of_any_batch_take_one_path():
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(10)
    B, Hkv, D, n = 40, 8, 128, 130
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    ki = torch.randint(0, 4096, (B, Hkv, n, 32), generator=gen, device="cuda", dtype=torch.int32)
    vi = torch.randint(0, 256, (B, Hkv, n, 16), generator=gen, device="cuda", dtype=torch.uint8)
    q, kcb, vcb = r(B, 2 * Hkv, 1, D), r(4096, 4), r(256, 8)
    out = K.vecinfer_attend_indices(q, ki, kcb, vi, vcb, 0.02, n_tokens=n)
    assert out is not None
    few = K.vecinfer_attend_indices(q[7:9], ki[7:9].contiguous(), kcb, vi[7:9].contiguous(), vcb, 0.02, n_tokens=n)
    # (the cut follows the batch: the sums' order differs, 130 tokens of unit variance)
    assert float((out[7:9] - few).abs().max()) < 1e-5
