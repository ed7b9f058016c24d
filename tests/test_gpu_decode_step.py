"""Decode steps in one launch: kv heads of 64 channels kept in pairs, and batches whose sequences differ in length,
each against the form with its arguments prepared by torch operations, bit for bit."""

import math

import pytest
import torch

from tests._gpu import gpu, require_gpu
from veloxquant_mlx_amd import kernels as K
from veloxquant_mlx_amd.cache import KVCacheConfig, KVCacheFactory, LayerStackedKIVICache
from veloxquant_mlx_amd.cache.kivi_cache import own_half_of_paired_output, pad_queries_for_paired_heads

pytestmark = gpu


def _cache(D, bits, g, B, H, ctx, dtype, seed, meta="float16", R=128):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda")
    c = KVCacheFactory.create(KVCacheConfig(method="kivi", head_dim=D, bit_width_inlier=bits, kivi_group_size=g, residual_length=R,
                                            fused_sdpa=True, fused_sdpa_memory_bound=True, kivi_meta_dtype=meta))
    f = torch.exp(rand(D))
    c.update_and_fetch((rand(B, H, ctx, D) * f).to(dtype), rand(B, H, ctx, D).to(dtype))
    return c, lambda: ((rand(B, H, 1, D) * f).to(dtype), rand(B, H, 1, D).to(dtype)), rand


@pytest.mark.parametrize("Hq,H,bits,g,B,ctx,dtype,meta", [
    (32, 8, 2, 32, 1, 700, torch.float16, "float16"), (32, 8, 4, 64, 3, 192, torch.bfloat16, "float16"),
    (14, 2, 4, 32, 2, 1000, torch.float16, "float16"), (9, 3, 3, 32, 2, 161, torch.bfloat16, "float16"),
    (5, 5, 2, 32, 1, 4099, torch.float16, "float32"), (40, 2, 4, 32, 1, 333, torch.float16, "float16"),
    (8, 8, 4, 32, 40, 200, torch.float16, "float16")])
def test_paired_heads_step_is_the_padded_one(Hq, H, bits, g, B, ctx, dtype, meta):
    """Queries read and outputs written by halves against queries padded with zeros and halves taken afterwards: the same
    bits under a fixed order, token after token across a flush, with the newest token brought along by the launch."""
    require_gpu()
    scale = 0.125
    a, new, rand = _cache(64, bits, g, B, H, ctx, dtype, Hq + ctx, meta)
    b, _, _ = _cache(64, bits, g, B, H, ctx, dtype, Hq + ctx, meta)
    deferred = 0
    for step in range(g + 2):
        k, v = new()
        for c in (a, b):
            c.update_and_fetch(k, v)
        q = rand(B, Hq, 1, 64).to(dtype)
        deferred += a._pending is not None
        got = a.fused_sdpa(q, scale, fixed_order=True)
        b._store_pending()
        kw = dict(causal=True, sliding_window=0, fixed_order=True, lengths=None, num_splits=0)
        want = own_half_of_paired_output(b._attend(pad_queries_for_paired_heads(q, H), scale, **kw), H)
        assert got.shape == q.shape and got.dtype == q.dtype and a._pending is None
        assert torch.equal(got, want), step
        n = a.offset - a._n_quantized
        assert torch.equal(a._tail_k[:, :, :n], b._tail_k[:, :, :n]) and torch.equal(a._tail_v[:, :, :n], b._tail_v[:, :, :n])
    assert deferred >= g - 1
    assert int(K._counters(q.device).abs().sum()) == 0


@pytest.mark.parametrize("D,Hq,H,bits,dtype", [(128, 32, 8, 4, torch.float16), (64, 9, 3, 2, torch.bfloat16), (64, 8, 4, 4, torch.float16),
                                               (256, 12, 4, 2, torch.bfloat16), (128, 6, 2, 8, torch.float16)])
def test_lengths_of_a_batch_in_the_launch(D, Hq, H, bits, dtype):
    """One length a sequence, clamped to prefix and tail inside the kernels, against the two clamped lists: the same bits, for
    lengths at every edge; the newest token is stored whether its sequence sees it or not."""
    require_gpu()
    B, g, ctx, scale = 9, 32, 700, 1 / math.sqrt(D)
    c, new, rand = _cache(D, bits, g, B, H, ctx, dtype, D + Hq)
    k, v = new()
    c.update_and_fetch(k, v)
    nq, total = c._n_quantized, c.offset
    lens = torch.tensor([0, 1, nq - 1, nq, nq + 1, total - 1, total, total + 5, 33], device="cuda")
    q = rand(B, Hq, 1, D).to(dtype)
    got = c.fused_sdpa(q, scale, lengths=lens, fixed_order=True)
    n_tail = total - nq
    pairs = k.shape[-1] == 64
    rows = c._tail_k[:, :, n_tail - 1]
    rows = rows.reshape(B, -1, 2, 64).reshape(B, -1, 64)[:, :H] if pairs else rows
    assert torch.equal(rows, k[:, :, 0])
    wide = pad_queries_for_paired_heads(q, H) if pairs else q
    want = K.kivi_packed_attend(wide, k_packed=c._kp, k_scale=c._ks, k_zero=c._kz, v_packed=c._vp, v_scale=c._vs, v_zero=c._vz,
                                n_packed=nq, bits=c._field, group_size=g, v_layout=c._v_layout, k_tail=c._tail_k,
                                v_tail=c._tail_v, n_tail=n_tail, scale=scale, out_dtype=dtype, fixed_order=True,
                                packed_lens=torch.clamp(lens, max=nq), tail_lens=torch.clamp(lens - nq, min=0, max=n_tail))
    want = own_half_of_paired_output(want, H) if pairs else want
    assert torch.equal(got, want)
    assert torch.equal(c.fused_sdpa(q, scale, lengths=lens.tolist(), fixed_order=True), want)                # host lengths
    assert torch.equal(c.fused_sdpa(q, scale, lengths=torch.stack([lens, lens], 1)[:, 0], fixed_order=True), want)   # strided ones
    # several query positions of such a batch (rows kernel, decode tiles or prefill blocks: whatever takes it)
    q = rand(B, Hq, 3, D).to(dtype)
    some = torch.clamp(lens, min=3)
    got = c.fused_sdpa(q, scale, lengths=some, fixed_order=True)
    alone = [c.fused_sdpa(q, scale, lengths=torch.full((B,), int(n), device="cuda"), fixed_order=True)[i] for i, n in enumerate(some)]
    assert torch.equal(got, torch.stack(alone))
    want = _clamped_lists(c, pad_queries_for_paired_heads(q, H) if pairs else q, some, scale)
    assert torch.equal(got, own_half_of_paired_output(want, H) if pairs else want)


@pytest.mark.parametrize("D,Hq,H,B,ctx,bits,dtype", [(128, 32, 8, 9, 4700, 2, torch.float16), (128, 14, 2, 26, 9000, 4, torch.bfloat16),
                                                     (64, 16, 16, 7, 6000, 2, torch.float16), (256, 12, 4, 7, 8700, 2, torch.bfloat16)])
def test_a_sequences_bits_do_not_depend_on_the_lengths_beside_it(D, Hq, H, B, ctx, bits, dtype):
    """Under a fixed order, of batches whose blocks are cut by all lengths otherwise: sequences of different lengths against batches
    whose sequences all have one of these lengths, bit for bit, and the cut by all lengths against the oracle's bar."""
    require_gpu()
    c, _, rand = _cache(D, bits, 32, B, H, ctx, dtype, D + B)
    q, scale = rand(B, Hq, 1, D).to(dtype), D ** -0.5
    lens = torch.tensor([c.offset - (i * 997) % (ctx - 1) for i in range(B)], device="cuda")
    got = c.fused_sdpa(q, scale, lengths=lens, fixed_order=True)
    for i, n in enumerate(lens.tolist()):
        alike = torch.full((B,), n, device="cuda")
        assert torch.equal(got[i], c.fused_sdpa(q, scale, lengths=alike, fixed_order=True)[i]), (i, n)
    lists = _clamped_lists(c, pad_queries_for_paired_heads(q, H) if D == 64 else q, lens, scale)
    assert torch.equal(got, own_half_of_paired_output(lists, H) if D == 64 else lists)
    on_demand = c.fused_sdpa(q, scale, lengths=lens, fixed_order=False)
    assert float((on_demand.float() - got.float()).abs().max()) < (2e-3 if dtype == torch.float16 else 1.6e-2)


@pytest.mark.parametrize("D,Hq,H,B,ctx,bits,Sq,window,dtype", [
    (128, 32, 8, 7, 5100, 2, 1, 0, torch.float16),         # a token brought along by the launch
    (128, 14, 2, 30, 4700, 4, 1, 0, torch.bfloat16),
    (64, 16, 16, 6, 5100, 2, 1, 0, torch.float16),         # heads of 64 channels in pairs
    (64, 9, 3, 26, 8300, 2, 1, 700, torch.bfloat16),       # an odd number of them, under a window
    (256, 12, 4, 7, 8700, 2, 1, 0, torch.bfloat16),
    (128, 8, 2, 13, 4800, 2, 4, 0, torch.float16),         # several positions, two row tiles a kv head
    (128, 32, 8, 2, 6000, 4, 6, 1000, torch.float16),      # and a window
    (128, 4, 1, 64, 4500, 2, 2, 0, torch.float16),         # as many sequences as one wave holds
    (256, 4, 1, 64, 4500, 2, 1, 0, torch.float16)])
def test_steps_over_evened_blocks(D, Hq, H, B, ctx, bits, Sq, window, dtype):
    """The cut by all lengths through the cache's own entry point: one int64 length a sequence, spread over the whole context, two steps
    with their tokens brought along where that is done, against the general kernel over the two clamped lists."""
    require_gpu()
    c, new, rand = _cache(D, bits, 32, B, H, ctx, dtype, D + B)
    scale = D ** -0.5
    lens = torch.tensor([c.offset - (i * 1009) % (ctx - Sq) for i in range(B)], device="cuda")
    for step in range(2):
        c.update_and_fetch(*new())
        lens += 1
        q = rand(B, Hq, Sq, D).to(dtype)
        got = c.fused_sdpa(q, scale, lengths=lens, sliding_window=window)
        wide = pad_queries_for_paired_heads(q, H) if D == 64 else q
        plan, shapes = {}, {}
        for fixed, out in ((False, plan), (True, shapes)):
            _clamped_lists(c, wide, lens, scale, window, fixed_order=fixed, _plan_out=out)
        assert plan["path"] == 1 and plan["nparts"] >= shapes["nparts"]
        want = _clamped_lists(c, wide, lens, scale, window, fixed_order=None, num_splits=-1)
        want = own_half_of_paired_output(want, H) if D == 64 else want
        # (two roundings of an output of up to 4: half a unit in the last place each)
        assert float((got.float() - want.float()).abs().max()) < (4e-3 if dtype == torch.float16 else 3.2e-2), step
    assert int(K._counters(q.device).abs().sum()) == 0


@pytest.mark.parametrize("D,Hq,H,B,ctx,bits", [(128, 32, 8, 7, 5100, 2), (128, 10, 2, 64, 4500, 4), (256, 12, 4, 7, 8700, 2)])
def test_protected_rows_over_evened_blocks(D, Hq, H, B, ctx, bits):
    """Protected rows are put in by a launch that reads all partials of a row: the cut by all lengths of the batch, whose shorter sequences
    have fewer of them, against the cut by the shapes, with NaN in the workspace beforehand."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(B)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").half()
    c = KVCacheFactory.create(KVCacheConfig(method="kivi_sink", head_dim=D, bit_width_inlier=bits, kivi_group_size=32, residual_length=128,
                                            n_sink_tokens=3, fused_sdpa=True))
    k = rand(B, H, ctx, D)
    k[:, :, [40, 3111]] *= 9
    c.update_and_fetch(k, rand(B, H, ctx, D))
    assert c._extra_attend_args()
    q, scale = rand(B, Hq, 1, D), D ** -0.5
    lens = torch.tensor([ctx - (i * 1009) % (ctx - 1) for i in range(B)], device="cuda")
    want = c.fused_sdpa(q, scale, lengths=lens, fixed_order=True)
    K._workspace(q.device, 1 << 20).fill_(0xff)
    got = c.fused_sdpa(q, scale, lengths=lens, fixed_order=False)
    assert torch.isfinite(want).all() and float((got.float() - want.float()).abs().max()) < 4e-3   # (two roundings of an output of up to 4)
    assert int(K._counters(q.device).abs().sum()) == 0


def test_a_stack_of_layers_of_different_lengths_over_evened_blocks():
    """Layers whose contexts differ in length as the sequences of one launch, on demand."""
    require_gpu()
    NL, B, H, D, dtype = 6, 1, 8, 128, torch.float16
    cfg = KVCacheConfig(method="kivi", head_dim=D, bit_width_inlier=2, kivi_group_size=32, residual_length=128, fused_sdpa=True,
                        fused_sdpa_memory_bound=True, fused_sdpa_max_ctx=8192)
    stack, gen = LayerStackedKIVICache(cfg, NL), torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").to(dtype)
    for l in range(NL):
        n = 8000 - 1303 * l
        stack[l].update_and_fetch(rand(B, H, n, D), rand(B, H, n, D))
    q = rand(NL, B, 32, 1, D)
    out = stack.fused_sdpa_all(q, 0.09)
    for l in range(NL):
        assert float((out[l].float() - stack[l].fused_sdpa(q[l], 0.09).float()).abs().max()) < 2e-3, l


def test_evened_blocks_in_a_graph_read_the_lengths_of_the_replay():
    """A captured step over uneven sequences, replayed after the lengths changed, between eager steps."""
    require_gpu()
    B, H, D, dtype = 7, 8, 128, torch.float16
    c, _, rand = _cache(D, 2, 32, B, H, 5100, dtype, 3)
    q, lens, out = rand(B, 32, 1, D).to(dtype), torch.full((B,), c.offset, device="cuda"), torch.empty(B, 32, 1, D, dtype=dtype, device="cuda")
    nq, n_tail = c._n_quantized, c.offset - c._n_quantized
    kw = dict(k_packed=c._kp, k_scale=c._ks, k_zero=c._kz, v_packed=c._vp, v_scale=c._vs, v_zero=c._vz, n_packed=nq, bits=c._field, group_size=32,
              v_layout=c._v_layout, k_tail=c._tail_k, v_tail=c._tail_v, n_tail=n_tail, scale=0.09)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            K.kivi_packed_attend(q, seq_lens=lens, out=out, **kw)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        K.kivi_packed_attend(q, seq_lens=lens, out=out, **kw)
    for step in range(4):
        lens.copy_(torch.tensor([max(1, c.offset - (i + step) * 811 * (step > 0)) for i in range(B)]))
        out.zero_()
        graph.replay()
        got = out.clone()
        eager = c.fused_sdpa(q, 0.09, lengths=lens)
        torch.cuda.synchronize()
        want = _clamped_lists(c, q, lens, 0.09, fixed_order=None, num_splits=-1)
        assert float((got.float() - want.float()).abs().max()) < 2e-3 and float((eager.float() - want.float()).abs().max()) < 2e-3, step


def test_uneven_lengths_in_the_built_in_scratch():
    """Shapes whose evened partials exceed the built-in scratch fall back to the cut with fewer; smaller ones are evened there as well."""
    require_gpu()
    for B, Hq, H, D, n in ((34, 40, 5, 256, 4128), (7, 16, 8, 128, 4352)):
        gen = torch.Generator(device="cuda").manual_seed(B)
        k, v = (torch.randn((B, H, n, D), generator=gen, device="cuda").half() for _ in range(2))
        q = torch.randn((B, Hq, 1, D), generator=gen, device="cuda").half()
        kp, ks, kz = K.kivi_quant_pack(k, -2, 32, 2, meta_dtype=torch.float16)
        vp, vs, vz = K.kivi_quant_pack(v, -1, 32, 2, meta_dtype=torch.float16, v_layout="token")
        lens = torch.tensor([n - (i * 613) % n for i in range(B)], dtype=torch.int32, device="cuda")
        kw = dict(k_packed=kp, k_scale=ks, k_zero=kz, v_packed=vp, v_scale=vs, v_zero=vz, n_packed=n, bits=2, group_size=32, v_layout="token",
                  k_tail=k[:, :, :70].contiguous(), v_tail=v[:, :, :70].contiguous(), n_tail=70, scale=D ** -0.5, out_dtype=torch.float32,
                  packed_lens=lens // 32 * 32, tail_lens=lens % 71)
        got = K.kivi_packed_attend(q, static_scratch=True, **kw)
        assert float((got - K.kivi_packed_attend(q, num_splits=-1, **kw)).abs().max()) < 2e-3


def _clamped_lists(c, q, lens, scale, window=0, **more):
    """The call with two clamped lists of lengths in place of one length a sequence."""
    nq, n_tail = c._n_quantized, c.offset - c._n_quantized
    kw = dict(k_packed=c._kp, k_scale=c._ks, k_zero=c._kz, v_packed=c._vp, v_scale=c._vs, v_zero=c._vz, n_packed=nq, bits=c._field,
              group_size=c._group_size, v_layout=c._v_layout) if nq else {}
    return K.kivi_packed_attend(q, k_tail=c._tail_k, v_tail=c._tail_v, n_tail=n_tail, scale=scale, causal=q.shape[2] > 1,
                                out_dtype=q.dtype, sliding_window=window, tiles=False, packed_lens=torch.clamp(lens, max=nq),
                                tail_lens=torch.clamp(lens - nq, min=0, max=n_tail), **{"fixed_order": True, **kw, **more})


@pytest.mark.parametrize("B,Hq,H,D,Sq,window,ctx,dtype", [
    (2, 64, 8, 128, 1, 1024, 16400, torch.float16), (7, 12, 4, 256, 1, 1024, 9000, torch.bfloat16), (2, 32, 8, 128, 4, 1024, 8200, torch.float16),
    (3, 12, 4, 128, 5, 300, 4100, torch.float16), (32, 32, 8, 128, 64, 0, 128, torch.float16), (5, 8, 2, 128, 40, 30, 100, torch.bfloat16)])
def test_lengths_and_a_window_from_an_empty_workspace(B, Hq, H, D, Sq, window, ctx, dtype):
    """Lengths a sequence beside a window, and a right-padded prompt over plain rows: the call finds the scratch of the launch that
    runs with no workspace left from earlier calls, and gives the bits of the two clamped lists."""
    require_gpu()
    c, new, rand = _cache(D, 4, 32, B, H, ctx, dtype, ctx + Sq)
    q, scale = rand(B, Hq, Sq, D).to(dtype), D ** -0.5
    lens = torch.tensor([max(Sq, c.offset - 37 * (i % 4)) for i in range(B)], device="cuda")
    K._workspaces.clear()
    got = c.fused_sdpa(q, scale, lengths=lens, sliding_window=window, fixed_order=True)
    assert torch.equal(got, _clamped_lists(c, q, lens, scale, window))
    k, v = new()
    c.update_and_fetch(k, v)   # a step on top, its token brought along where that is done
    q, lens = rand(B, Hq, 1, D).to(dtype), lens + 1
    K._workspaces.clear()
    got = c.fused_sdpa(q, scale, lengths=lens, sliding_window=window, fixed_order=True)
    assert torch.equal(got, _clamped_lists(c, q, lens, scale, window))


def test_pair_heads_refusals():
    """What the launch for pairs does not take is refused before anything is written."""
    require_gpu()
    c, new, rand = _cache(64, 4, 32, 1, 4, 300, torch.float16, 3)
    nq = c._n_quantized
    kw = dict(k_packed=c._kp, k_scale=c._ks, k_zero=c._kz, v_packed=c._vp, v_scale=c._vs, v_zero=c._vz, n_packed=nq, bits=4,
              group_size=32, v_layout="token", k_tail=c._tail_k, v_tail=c._tail_v, n_tail=c.offset - nq, scale=0.1)
    ok = rand(1, 8, 1, 64).half()
    for q, extra in ((rand(1, 8, 2, 64).half(), {}), (rand(1, 6, 1, 64).half(), {}), (rand(1, 8, 1, 128).half(), {}),
                     (ok, dict(static_scratch=True)), (ok, dict(_single_launch=False)), (ok, dict(num_splits=-1)),
                     (ok, dict(seq_lens=torch.tensor([5], dtype=torch.int32, device="cuda")))):
        with pytest.raises(ValueError):
            K.kivi_packed_attend(q, pair_heads=4, **{**kw, **extra})
    with pytest.raises(ValueError):
        K.kivi_packed_attend(ok, pair_heads=8, **kw)


@pytest.mark.parametrize("D,Hq,H,bits,g,meta,dtype", [(128, 8, 2, 2, 32, "float16", torch.bfloat16), (128, 3, 3, 4, 128, "float16", torch.float16),
                                                      (64, 16, 4, 2, 64, "float32", torch.float16), (256, 12, 4, 4, 32, "float16", torch.float16)])
@pytest.mark.parametrize("units", [1, 2, 11, 12, 13, 24, 47, 48, 49, 59, 60, 61, 73])
def test_units_dealt_over_the_waves_of_one_block(D, Hq, H, bits, g, meta, dtype, units):
    """One block a kv head (num_splits=1) over numbers of 32-token units around one chunk a wave, where they are dealt out
    evenly, and beyond, where waves draw chunks: against the general kernel, which sums token by token in float32.  Output
    rounding is 2^-11 (fp16) or 2^-8 (bf16) of values of order one, the products' remainder terms 2^-21; the
    cache's own call is the same bits as the general wrapper's."""
    require_gpu()
    ctx = 128 + -(-32 * units // g) * g
    c, new, rand = _cache(D, bits, g, 2, H, ctx, dtype, units, meta)
    q = rand(2, Hq, 1, D).to(dtype)
    got = c.fused_sdpa(q, D ** -0.5, fixed_order=True, num_splits=1)
    kw = dict(k_packed=c._kp, k_scale=c._ks, k_zero=c._kz, v_packed=c._vp, v_scale=c._vs, v_zero=c._vz, n_packed=c._n_quantized,
              bits=c._field, group_size=g, v_layout=c._v_layout, k_tail=c._tail_k, v_tail=c._tail_v, n_tail=c.offset - c._n_quantized,
              scale=D ** -0.5)
    wide = q if D > 64 else pad_queries_for_paired_heads(q, H)
    half = (lambda o: o) if D > 64 else (lambda o: own_half_of_paired_output(o, H))
    assert torch.equal(got, half(K.kivi_packed_attend(wide, fixed_order=True, num_splits=1, **kw)))
    want = half(K.kivi_packed_attend(wide.float(), num_splits=-1, out_dtype=torch.float32, **kw))
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert float((got.float() - want).abs().max()) <= eps * float(want.abs().max()) + 1e-3
    free = c.fused_sdpa(q, D ** -0.5)
    assert float((free.float() - want).abs().max()) <= eps * float(want.abs().max()) + 1e-3


@pytest.mark.parametrize("D,Hq,H,bits,g,B,ctx,dtype,meta", [
    (256, 12, 4, 2, 32, 3, 700, torch.bfloat16, "float16"), (256, 8, 4, 4, 64, 1, 193, torch.float16, "float32"),
    (256, 10, 1, 3, 128, 2, 1100, torch.float16, "float16"), (64, 9, 3, 2, 32, 3, 700, torch.bfloat16, "float16"),
    (64, 10, 5, 4, 64, 1, 193, torch.float16, "float32")])
def test_step_takes_its_token_at_once(D, Hq, H, bits, g, B, ctx, dtype, meta):
    """A caller that writes its key and value buffers again between a step's update and its attention: the same bits as with
    tensors of its own a step, token after token across a flush."""
    require_gpu()
    a, new, rand = _cache(D, bits, g, B, H, ctx, dtype, Hq + ctx, meta)
    b, _, _ = _cache(D, bits, g, B, H, ctx, dtype, Hq + ctx, meta)
    kbuf, vbuf = (torch.empty(B, H, 1, D, dtype=dtype, device="cuda") for _ in range(2))
    for step in range(g + 2):
        k, v = new()
        b.update_and_fetch(k, v)
        a.update_and_fetch(kbuf.copy_(k), vbuf.copy_(v))
        kbuf.fill_(55.0), vbuf.fill_(-77.0)
        q = rand(B, Hq, 1, D).to(dtype)
        kw = dict(fixed_order=True, sliding_window=0 if step % 3 else 150)
        assert torch.equal(a.fused_sdpa(q, D ** -0.5, **kw), b.fused_sdpa(q, D ** -0.5, **kw)), step
        n = a.offset - a._n_quantized
        assert torch.equal(a._tail_k[:, :, :n], b._tail_k[:, :, :n]) and torch.equal(a._tail_v[:, :, :n], b._tail_v[:, :, :n])


@pytest.mark.parametrize("how", ["attend", "general", "trim", "stack"])
def test_attention_on_another_stream_keeps_the_tokens_memory(how, monkeypatch):
    """A token handed over on one stream and read by a launch on another: its memory is held for that stream; on the same
    stream nothing is recorded."""
    require_gpu()
    held = []
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: held.append((t.data_ptr(), s.cuda_stream)))
    H, D, ctx = 4, 128, 400
    if how == "stack":
        cfg = KVCacheConfig(method="kivi", head_dim=D, bit_width_inlier=4, kivi_group_size=32, fused_sdpa=True, fused_sdpa_memory_bound=True)
        c = LayerStackedKIVICache(cfg, 2)
        layers = c.layers
        for l in layers:
            l.update_and_fetch(*(torch.randn(1, H, ctx, D, device="cuda").half() for _ in range(2)))
        c.fused_sdpa_all(torch.randn(2, 1, 8, 1, D, device="cuda").half(), 0.1)
    else:
        c, _, _ = _cache(D, 4, 32, 1, H, ctx, torch.float16, 1)
        layers = [c]
    use = {"attend": lambda: c.fused_sdpa(torch.randn(1, 8, 1, D, device="cuda").half(), 0.1),
           "general": lambda: c.fused_sdpa(torch.randn(1, 8, 2, D, device="cuda").half(), 0.1),
           "trim": lambda: c.trim(0), "stack": lambda: c.fused_sdpa_all(torch.randn(2, 1, 8, 1, D, device="cuda").half(), 0.1)}[how]
    other = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), other):
        tokens = [[torch.randn(1, H, 1, D, device="cuda").half() for _ in range(2)] for _ in layers]
        for l, (k, v) in zip(layers, tokens):
            l.update_and_fetch(k, v)
            assert l._pending is not None
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            use()
        assert all(l._pending is None for l in layers)
        want = [(t.data_ptr(), other.cuda_stream) for kv in tokens for t in kv] if stream is other else []
        assert sorted(held) == sorted(want)
        torch.cuda.synchronize()


@pytest.mark.parametrize("D,bits,g,dtype,more,deferred", [
    (128, 4, 32, torch.float16, {}, True), (128, 1, 64, torch.bfloat16, {}, True), (64, 2, 32, torch.float16, {}, True),
    (128, 8, 32, torch.float16, {}, False), (128, 3, 32, torch.float16, dict(kivi_code_field="tight"), False),
    (128, 4, 32, torch.float16, dict(kivi_value_layout="channel"), False), (128, 4, 32, torch.float32, {}, False),
    (128, 4, 16, torch.bfloat16, {}, False), (64, 8, 32, torch.float16, {}, False), (64, 4, 32, torch.float16, dict(kivi_pair_heads=False), False)])
def test_only_a_launch_that_stores_the_token_is_left_it(D, bits, g, dtype, more, deferred, monkeypatch):
    """A step's token waits for the attention launch only where that launch stores it, and the step is one library call either way:
    none is refused and made again."""
    require_gpu()
    B, H, Hq = 2, 4, 8
    c = KVCacheFactory.create(KVCacheConfig(method="kivi", head_dim=D, bit_width_inlier=bits, kivi_group_size=g, residual_length=64,
                                            fused_sdpa=True, fused_sdpa_memory_bound=True, **more))
    r = lambda *s: torch.randn(s, device="cuda").to(dtype)
    c.update_and_fetch(r(B, H, 64 + 2 * g + 3, D), r(B, H, 64 + 2 * g + 3, D))
    taken, real = [], K.kivi_decode_attend
    monkeypatch.setattr(K, "kivi_decode_attend", lambda *a: taken.append(real(*a)) or taken[-1])
    k, v = r(B, H, 1, D), r(B, H, 1, D)
    c.update_and_fetch(k, v)
    assert (c._pending is not None) == deferred
    out = c.fused_sdpa(r(B, Hq, 1, D), 0.1)
    assert c._pending is None and out.shape == (B, Hq, 1, D) and len(taken) == 1 and taken[0] is not None
    row = c._tail_k[:, :, c.offset - c._n_quantized - 1]
    assert torch.equal(row.reshape(B, H, D), k[:, :, 0])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,Hq,H,S", [(64, 8, 4, 1), (64, 9, 3, 1), (128, 8, 2, 1), (128, 4, 1, 3), (256, 12, 4, 1)])
@pytest.mark.parametrize("off", [1, 3, 4, 8])
def test_queries_between_sixteen_byte_boundaries(D, Hq, H, S, dtype, off):
    """Queries that are a contiguous view at an odd place: the bits that aligned ones give."""
    require_gpu()
    c, new, rand = _cache(D, 4, 32, 2, H, 300, torch.float16, D + off)
    q = rand(2, Hq, S, D).to(dtype)
    moved = torch.zeros(q.numel() + off, dtype=dtype, device="cuda")[off:].view(q.shape).copy_(q)
    assert moved.is_contiguous() and torch.equal(c.fused_sdpa(moved, 0.1, fixed_order=True), c.fused_sdpa(q, 0.1, fixed_order=True))


def test_numbers_that_the_packed_block_does_not_hold():
    """A scale past float32 and a split count past 32 bits go the general way, as they did before steps had a block of their own."""
    require_gpu()
    c, new, rand = _cache(128, 4, 32, 1, 2, 300, torch.float16, 5)
    q = rand(1, 4, 1, 128).half()
    assert c.fused_sdpa(q, 1e39).shape == q.shape
    # (kept as its low 32 bits: one run)
    assert torch.equal(c.fused_sdpa(q, 0.1, num_splits=(1 << 32) + 1, fixed_order=True), c.fused_sdpa(q, 0.1, num_splits=1, fixed_order=True))


def test_a_tail_unit_without_a_number_counts_for_nothing():
    """32 tail tokens whose fp16 keys are no numbers, one unit of a wave of its own: the attention over all other slots (values of
    order one; weights in fp16 and the output's rounding, 2^-11)."""
    require_gpu()
    B, Hq, H, D, scale, dtype = 1, 8, 2, 128, 128 ** -0.5, torch.float16
    c, new, rand = _cache(D, 4, 32, B, H, 300, dtype, 11)
    nq, n_tail = c._n_quantized, c.offset - c._n_quantized
    q = rand(B, Hq, 1, D).to(dtype)
    c._tail_k[:, :, 32:64] = float("nan")
    keep = [i for i in range(c.offset) if not nq + 32 <= i < nq + 64]
    deq = lambda p, s, z, axis, kw: K.kivi_dequant(p, s, z, axis, 32, c._field, nq, D, out_dtype=torch.float32, **kw)
    k = torch.cat([deq(c._kp, c._ks, c._kz, -2, {}), c._tail_k[:, :, :n_tail].float()], 2)[:, :, keep].repeat_interleave(Hq // H, 1)
    v = torch.cat([deq(c._vp, c._vs, c._vz, -1, dict(v_layout=c._v_layout)), c._tail_v[:, :, :n_tail].float()], 2)[:, :, keep].repeat_interleave(Hq // H, 1)
    want = torch.softmax((q.float() * k).sum(-1) * scale, -1)[..., None].mul(v).sum(2, keepdim=True)
    got = c.fused_sdpa(q, scale).float()
    assert float((got - want).abs().max()) <= 2.0 ** -11 * float(want.abs().max()) + 2e-3


@pytest.mark.parametrize("D,Hq,H,ctx", [(128, 32, 8, 1500), (64, 8, 4, 700), (256, 8, 2, 900)])
def test_workspace_aligned_as_floats_are(D, Hq, H, ctx, monkeypatch):
    """A workspace four bytes off a boundary of eight: the bits of an aligned one, with the merge in the launch and after it."""
    require_gpu()
    c, new, rand = _cache(D, 4, 32, 1, H, ctx, torch.float16, ctx)
    q = rand(1, Hq, 1, D).half()
    want = c.fused_sdpa(q, 0.1, fixed_order=True)
    room = torch.empty(8 << 20, dtype=torch.uint8, device="cuda")[4:]
    assert room.data_ptr() % 8 == 4
    monkeypatch.setattr(K, "_workspace", lambda *a: room)
    assert torch.equal(c.fused_sdpa(q, 0.1, fixed_order=True), want)
    if D != 64:
        kw = dict(k_packed=c._kp, k_scale=c._ks, k_zero=c._kz, v_packed=c._vp, v_scale=c._vs, v_zero=c._vz, n_packed=c._n_quantized,
                  bits=c._field, group_size=32, v_layout=c._v_layout, k_tail=c._tail_k, v_tail=c._tail_v, n_tail=c.offset - c._n_quantized,
                  scale=0.1, fixed_order=True)
        assert torch.equal(K.kivi_packed_attend(q, _single_launch=False, **kw), want)
