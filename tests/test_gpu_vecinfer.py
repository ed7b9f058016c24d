"""HIP VecInfer assignment / gather against the CPU oracle: indices bit-exact
(float32 distances, left-to-right sum, lowest index on ties).  Restates
veloxquant_mlx/tests/cache/test_vecinfer_metal_parity.py:140-167 and the shapes
of blogs/metal-kernels.md:150-157."""

import numpy as np
import pytest
import torch

from oracle import cref, vecinfer as ov
from tests._gpu import gpu, host, require_gpu, to_dev
from veloxquant_mlx_amd import kernels as K
from veloxquant_mlx_amd.allocators.vecinfer import walsh_hadamard_matrix
from veloxquant_mlx_amd.cache import KVCacheConfig, KVCacheFactory

pytestmark = gpu


def _keys(shape, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(shape).astype(np.float32)
    return (x * np.exp(rng.standard_normal(shape[-1])).astype(np.float32)).astype(np.float16), rng


@pytest.mark.parametrize("sub,nc,D", [(8, 256, 256), (4, 256, 128), (4, 4096, 128), (2, 16, 64), (16, 64, 128),
                                      (3, 50, 96), (1, 7, 8)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
def test_assign_bit_exact(sub, nc, D, dtype):
    require_gpu()
    x, rng = _keys((2, 3, 37, D), seed=sub * 1000 + nc)
    cb = rng.standard_normal((nc, sub)).astype(np.float16)
    xt, cbt = to_dev(x, dtype), to_dev(cb)
    got = K.vecinfer_quantize_metal(xt, cbt, sub)
    assert got.dtype == torch.int32 and got.shape == (2, 3, 37, D // sub)
    ref = ov.quantize_vq(host(xt), cb, sub)
    np.testing.assert_array_equal(host(got), ref)
    if nc <= 256:
        got8 = K.vecinfer_quantize_metal(xt, cbt, sub, index_dtype=torch.uint8)
        np.testing.assert_array_equal(host(got8), ref.astype(np.uint8))


def test_exact_ties_take_the_lowest_index():
    require_gpu()
    rng = np.random.default_rng(1)
    cb = rng.standard_normal((64, 8)).astype(np.float32)
    cb[40] = cb[9]
    cb[63] = cb[9]
    x = np.tile(cb[9], (100, 1)) + rng.standard_normal((100, 8)).astype(np.float32) * 1e-3
    got = host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), 8))
    assert set(got.reshape(-1).tolist()) == {9}
    # symmetric tie: x exactly between two centroids along one axis
    cb2 = np.zeros((4, 2), np.float32)
    cb2[1] = [2, 0]; cb2[2] = [0, 2]; cb2[3] = [2, 2]
    x2 = np.array([[1, 0], [0, 1], [1, 1], [2, 1]], np.float32)
    got2 = host(K.vecinfer_quantize_metal(to_dev(x2), to_dev(cb2), 2)).reshape(-1)
    np.testing.assert_array_equal(got2, ov.quantize_vq(x2, cb2, 2).reshape(-1))
    assert got2.tolist() == [0, 0, 0, 1]


def test_config2_falcon_shape_full_size():
    """keys [4,4096,256] fp16 with outlier channels, 256 fp16 centroids of 8 dims:
    524,288 sub-vectors, every index equal to the brute-force C oracle."""
    require_gpu()
    x, rng = _keys((4, 4096, 256), seed=2)
    cb = rng.standard_normal((256, 8)).astype(np.float16)
    got = host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), 8, index_dtype=torch.uint8))
    ref = cref.vq_assign(x.astype(np.float32), cb.astype(np.float32), 8)
    assert got.shape == (4, 4096, 32)
    np.testing.assert_array_equal(got, ref.astype(np.uint8))
    # the numpy restatement agrees on a slice, with the near-tie census the parity report quotes
    sl, margin = ov.quantize_vq(x[:1, :512], cb, 8, return_margin=True)
    np.testing.assert_array_equal(got[:1, :512], sl.astype(np.uint8))
    print(f"near-ties (<= 4 ulp of the best distance): {(margin <= 4 * np.spacing(np.float32(8.0))).sum()} of {margin.size}")


def test_dequant_gather_and_clamp():
    require_gpu()
    rng = np.random.default_rng(3)
    cb = rng.standard_normal((256, 8)).astype(np.float32)
    idx = rng.integers(0, 256, size=(2, 5, 16)).astype(np.int32)
    out = K.vecinfer_dequant_metal(to_dev(idx), to_dev(cb))
    np.testing.assert_array_equal(host(out), ov.dequantize_vq(idx, cb))
    out16 = K.vecinfer_dequant_metal(to_dev(idx.astype(np.uint8)), to_dev(cb), out_dtype=torch.float16)
    np.testing.assert_array_equal(host(out16), ov.dequantize_vq(idx, cb).astype(np.float16))
    bad = idx.copy(); bad[0, 0, 0] = 9999
    outc = host(K.vecinfer_dequant_metal(to_dev(bad), to_dev(cb)))
    np.testing.assert_array_equal(outc[0, 0, :8], cb[255])


def test_round_trip_idempotent_at_scale():
    """assign(gather(assign(x))) == assign(x) whenever centroids are distinct."""
    require_gpu()
    x, rng = _keys((2, 2048, 128), seed=4)
    cb = to_dev(rng.standard_normal((256, 4)).astype(np.float16))
    i1 = K.vecinfer_quantize_metal(to_dev(x), cb, 4)
    i2 = K.vecinfer_quantize_metal(K.vecinfer_dequant_metal(i1, cb), cb, 4)
    assert torch.equal(i1, i2)


def test_wrapper_errors():
    require_gpu()
    x = to_dev(np.zeros((4, 10), np.float16))
    cb = to_dev(np.zeros((8, 4), np.float16))
    with pytest.raises(ValueError, match="not divisible by sub_dim"):
        K.vecinfer_quantize_metal(x, cb, 4)
    with pytest.raises(ValueError, match=r"codebook must be \[n_centroids, 5\]"):
        K.vecinfer_quantize_metal(x, cb, 5)
    with pytest.raises(ValueError, match="codebook must be 2D"):
        K.vecinfer_dequant_metal(to_dev(np.zeros((2, 2), np.int32)), cb.reshape(-1))


# ------------------------------------------------ the MFMA filter's undecided cases
@pytest.mark.parametrize("sub,nc", [(8, 256), (8, 200), (4, 256), (8, 5), (4, 17)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
def test_mfma_filter_near_ties_follow_the_exact_rule(sub, nc, dtype):
    """Sub-vectors placed (almost) on the bisector of two or more centroids, where only the
    float32 rounding of the sequential rule decides: one ulp nudges either way, clusters of
    near-identical centroids, exact duplicates in several tracker positions."""
    require_gpu()
    rng = np.random.default_rng(sub * 7 + nc)
    cb = rng.standard_normal((nc, sub)).astype(np.float16).astype(np.float32)
    if nc >= 17:
        cb[3] = cb[16]; cb[nc - 1] = cb[16]            # triple duplicate across tiles and rows
        cb[5] = cb[4] + np.float32(2.0 ** -10)           # a cluster of near-identical centroids
        cb[6] = cb[4] - np.float32(2.0 ** -10)
        cb[7] = cb[4]
    cbt = to_dev(cb, torch.float32 if dtype == torch.float32 else torch.float16)
    cbh = host(cbt).astype(np.float32)
    n = 4096 + 37
    a = rng.integers(0, nc, n)
    b = rng.integers(0, nc, n)
    mid = 0.5 * (cbh[a] + cbh[b])
    x = mid + rng.standard_normal((n, sub)).astype(np.float32) * np.float32(1e-4) * (rng.integers(0, 3, (n, 1)) > 0)
    x[::5] = cbh[a[::5]]                                 # exactly on a centroid (duplicates tie)
    xt = to_dev(x.astype(np.float32), dtype)
    got = host(K.vecinfer_quantize_metal(xt, cbt, sub)).reshape(-1)
    ref = ov.quantize_vq(host(xt).astype(np.float32), cbh, sub).reshape(-1)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("sub,nc", [(4, 513), (4, 1000), (4, 4095), (4, 4096), (8, 545), (8, 2047), (8, 2048)])
@pytest.mark.parametrize("n", [1, 65, 32768, 32769, 70001])
def test_large_codebooks_split_and_image_forms(sub, nc, n):
    """Codebooks above 512 centroids on both sides of the sub-vector count where the two forms of the kernel meet, with a
    partly filled last tile, duplicated and clustered centroids, sub-vectors on centroids and on bisectors, far outside the
    codebook, zeros and a NaN row (no distance below infinity: index 0)."""
    require_gpu()
    rng = np.random.default_rng(nc * 3 + n)
    cb = (rng.standard_normal((nc, sub)) * 3).astype(np.float32)
    cb[nc - 1] = cb[7]; cb[300] = cb[7]; cb[17] = cb[16] + np.float32(2.0 ** -12); cb[18] = cb[16]
    x = (rng.standard_normal((n, sub)) * 3).astype(np.float32)
    a, b = rng.integers(0, nc, n), rng.integers(0, nc, n)
    x[::7] = 0.5 * (cb[a[::7]] + cb[b[::7]])
    x[3::11] = cb[a[3::11]]
    x[5::1009] *= np.float32(3000)                   # outside the filter's range
    x[6::4001] = 0
    x[2::2003] = cb[7] + np.float32(1e-4)
    got = host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), sub)).reshape(-1)
    np.testing.assert_array_equal(got, cref.vq_assign(x, cb, sub).reshape(-1))
    x[0, 1] = np.nan
    assert host(K.vecinfer_quantize_metal(to_dev(x[:2]), to_dev(cb), sub)).reshape(-1)[0] == 0


@pytest.mark.parametrize("nc", [1, 2, 16, 31, 33, 63, 65, 97, 500, 513, 577, 1025])
@pytest.mark.parametrize("sub", [4, 8])
def test_rows_past_the_end_of_a_codebook_never_count(sub, nc):
    """Codebooks that end inside a tile, or leave the second tile of a pair empty: sub-vectors at the last centroid, at the origin
    with the codebook far from it, and out to the end of the filter's range (256 times the largest centroid) and past it."""
    require_gpu()
    rng = np.random.default_rng(nc * 10 + sub)
    cb = (rng.standard_normal((nc, sub)) + (6 if nc % 2 else 0)).astype(np.float32)
    x = np.concatenate([cb[-1] + rng.standard_normal((300, sub)) * 0.1, np.tile(cb[-1], (5, 1)), np.zeros((5, sub)),
                        rng.standard_normal((300, sub)) * np.abs(cb).max() * np.exp(rng.uniform(0, 7, (300, 1)))]).astype(np.float32)
    got = host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), sub)).reshape(-1)
    np.testing.assert_array_equal(got, cref.vq_assign(x, cb, sub).reshape(-1))


@pytest.mark.parametrize("far_out", [1e16, 3e19, float("inf")])
@pytest.mark.parametrize("sub,nc,n", [(4, 256, 200), (8, 300, 200), (4, 1000, 200), (4, 4096, 200), (8, 2048, 200), (4, 4096, 33000)])
def test_a_diverged_centroid_leaves_the_exact_rule_to_the_others(sub, nc, n, far_out):
    """One centroid whose square leaves the range the filter can be brought to, beside centroids whose squares pass the
    largest fp16 number: sub-vectors on and near all of them, in every form of the kernel."""
    require_gpu()
    rng = np.random.default_rng(nc + sub)
    cb = (rng.standard_normal((nc, sub)) * 300).astype(np.float32)
    cb[nc // 3] = far_out
    near = cb[rng.integers(0, nc, n)]
    near[~(np.abs(near[:, 0]) < 1e10)] = 5.0
    x = (near + rng.standard_normal((n, sub)) * np.float32(20) * (rng.random((n, 1)) < 0.7)).astype(np.float32)
    with np.errstate(all="ignore"):
        ref = cref.vq_assign(x, cb, sub).reshape(-1)
    np.testing.assert_array_equal(host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), sub)).reshape(-1), ref)


@pytest.mark.parametrize("scale", [1e-6, 1e-3, 1e3, 1e6])
def test_assignment_follows_the_exact_rule_at_any_scale(scale):
    require_gpu()
    rng = np.random.default_rng(3)
    for sub, nc, n in ((4, 4096, 500), (8, 256, 3000), (4, 1024, 40000)):
        cb = (rng.standard_normal((nc, sub)) * scale).astype(np.float32)
        x = (rng.standard_normal((n, sub)) * scale * np.exp(rng.standard_normal((n, 1)))).astype(np.float32)
        got = host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), sub)).reshape(-1)
        np.testing.assert_array_equal(got, cref.vq_assign(x, cb, sub).reshape(-1))


def test_mfma_filter_large_magnitudes_and_ragged_count():
    require_gpu()
    rng = np.random.default_rng(11)
    cb = (rng.standard_normal((256, 8)) * 30).astype(np.float16)
    for n in (1, 63, 64, 65, 1000):
        x = (rng.standard_normal((n, 8)) * np.exp(2 * rng.standard_normal(8))).astype(np.float16)
        got = host(K.vecinfer_quantize_metal(to_dev(x), to_dev(cb), 8)).reshape(-1)
        np.testing.assert_array_equal(got, ov.quantize_vq(x, cb, 8).reshape(-1))


# ---------------------------------------------------------------------------
# attention straight from the indices (look-up table + centroid histogram)
# ---------------------------------------------------------------------------

LUT_TOL = 2e-3   # max-abs against the float64 oracle; the reference's own bar is 1e-2
                 # (veloxquant_mlx/tests/cache/test_vecinfer_fused_sdpa.py:20)


def _lut_case(B, Hq, Hkv, Sq, S, D, sub_k, sub_v, C, seed, idx_dtype=np.uint8, cap=None, q_scale=1.0):
    rng = np.random.default_rng(seed)
    cap = cap or S
    q = (rng.standard_normal((B, Hq, Sq, D)) * q_scale).astype(np.float32)
    kcb = rng.standard_normal((C, sub_k)).astype(np.float32)
    vcb = rng.standard_normal((C, sub_v)).astype(np.float32)
    ki = rng.integers(0, C, (B, Hkv, cap, D // sub_k)).astype(idx_dtype)
    vi = rng.integers(0, C, (B, Hkv, cap, D // sub_v)).astype(idx_dtype)
    return q, ki, kcb, vi, vcb


def _lut_run(q, ki, kcb, vi, vcb, scale, q_dtype=torch.float32, cb_dtype=torch.float32, **kw):
    return host(K.metal_fused_sdpa(to_dev(q, q_dtype), to_dev(ki), to_dev(kcb, cb_dtype), to_dev(vi),
                                   to_dev(vcb, cb_dtype), scale, **kw)).astype(np.float32)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,S,D,sub,C", [
    (1, 4, 4, 1, 128, 64, 4, 256),       # the reference's default case (test_vecinfer_fused_sdpa.py:120-131)
    (1, 32, 8, 1, 256, 128, 8, 256),     # GQA 32/8 (ibid. 172-184)
    (1, 4, 4, 8, 128, 64, 4, 256),       # S_q = 8 (ibid. 218-228)
    (1, 4, 4, 1, 4096, 64, 4, 256),      # long context (ibid. 206-216)
    (2, 8, 2, 5, 777, 128, 8, 256),      # ragged length, several query rows per kv head
    (1, 8, 8, 1, 1500, 256, 16, 200),    # D = 256, fewer centroids
    (1, 2, 1, 3, 300, 96, 8, 17),        # n_sub = 12
])
def test_lut_attention_matches_the_gather_oracle(B, Hq, Hkv, Sq, S, D, sub, C, causal):
    require_gpu()
    q, ki, kcb, vi, vcb = _lut_case(B, Hq, Hkv, Sq, S, D, sub, sub, C, seed=S + D + Sq)
    scale = 1.0 / np.sqrt(D)
    ref = ov.fused_sdpa(q, ki, kcb, vi, vcb, scale, causal=causal)
    got = _lut_run(q, ki, kcb, vi, vcb, scale, causal=causal)
    assert got.shape == ref.shape
    assert np.max(np.abs(got - ref)) < LUT_TOL
    # 32-bit indices take the word path; same answer
    got32 = _lut_run(q, ki.astype(np.int32), kcb, vi.astype(np.int32), vcb, scale, causal=causal)
    assert np.max(np.abs(got32 - ref)) < LUT_TOL


@pytest.mark.parametrize("S", [1, 2])
def test_lut_attention_one_and_two_tokens(S):
    """veloxquant_mlx/tests/cache/test_vecinfer_fused_sdpa.py:186-204"""
    require_gpu()
    q, ki, kcb, vi, vcb = _lut_case(1, 4, 4, 1, S, 64, 4, 4, 256, seed=S)
    ref = ov.fused_sdpa(q, ki, kcb, vi, vcb, 0.125)
    assert np.max(np.abs(_lut_run(q, ki, kcb, vi, vcb, 0.125) - ref)) < LUT_TOL
    if S == 1:   # one token: the output is that token's value, whatever the query
        np.testing.assert_allclose(_lut_run(q, ki, kcb, vi, vcb, 0.125), ov.dequantize_vq(vi, vcb)[:, :, :1], atol=1e-6)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Sq,S,window", [(1, 256, 64), (8, 256, 64), (4, 1300, 100), (3, 40, 64), (2, 600, 1)])
def test_lut_attention_sliding_window(Sq, S, window, causal):
    """window mask of veloxquant_mlx/tests/cache/test_vecinfer_fused_sdpa.py:105-113, 155-170"""
    require_gpu()
    q, ki, kcb, vi, vcb = _lut_case(1, 4, 2, Sq, S, 64, 4, 4, 256, seed=window + Sq)
    ref = ov.fused_sdpa(q, ki, kcb, vi, vcb, 0.125, causal=causal, sliding_window=window)
    got = _lut_run(q, ki, kcb, vi, vcb, 0.125, causal=causal, sliding_window=window)
    assert np.max(np.abs(got - ref)) < LUT_TOL
    if window == 1 and causal:   # each query sees only its own position
        vh = ov.dequantize_vq(vi, vcb)
        np.testing.assert_allclose(got[0, 0], vh[0, 0, S - Sq:], atol=1e-6)


def test_lut_attention_mixed_sub_dims_dtypes_and_a_prefix_of_the_buffer():
    require_gpu()
    # keys in 8-wide, values in 4-wide sub-vectors; only the first 333 of 512 rows are tokens
    q, ki, kcb, vi, vcb = _lut_case(2, 8, 4, 2, 333, 128, 8, 4, 64, seed=5, cap=512)
    scale = 0.1
    ref = ov.fused_sdpa(q, ki[:, :, :333], kcb, vi[:, :, :333], vcb, scale)
    assert np.max(np.abs(_lut_run(q, ki, kcb, vi, vcb, scale, n_tokens=333) - ref)) < LUT_TOL
    # fp16 queries, codebooks and output: compare on the rounded operands
    q16, kcb16, vcb16 = (x.astype(np.float16).astype(np.float32) for x in (q, kcb, vcb))
    ref16 = ov.fused_sdpa(q16, ki[:, :, :333], kcb16, vi[:, :, :333], vcb16, scale)
    got16 = _lut_run(q, ki, kcb, vi, vcb, scale, q_dtype=torch.float16, cb_dtype=torch.float16, n_tokens=333)
    assert np.max(np.abs(got16 - ref16)) < LUT_TOL
    gotbf = host(K.metal_fused_sdpa(to_dev(q16), to_dev(ki), to_dev(kcb16), to_dev(vi), to_dev(vcb16), scale,
                                    n_tokens=333, out_dtype=torch.bfloat16).float())
    assert np.max(np.abs(gotbf - ref16)) < 2e-2   # bf16 output rounding


def test_lut_attention_properties():
    require_gpu()
    q, ki, kcb, vi, vcb = _lut_case(1, 8, 2, 4, 2000, 128, 8, 8, 256, seed=9)
    scale = 1.0 / np.sqrt(128)
    base = _lut_run(q, ki, kcb, vi, vcb, scale)
    # the token split must not matter
    for ns in (1, 2, 3, 4):
        assert np.max(np.abs(_lut_run(q, ki, kcb, vi, vcb, scale, num_splits=ns) - base)) < 1e-4
    # causal: the first query position cannot see the last three tokens
    ki2, vi2 = ki.copy(), vi.copy()
    ki2[:, :, -3:] += 7      # uint8 wraps inside the 256 centroids
    vi2[:, :, -3:] += 11
    pert = _lut_run(q, ki2, kcb, vi2, vcb, scale)
    assert np.max(np.abs(pert[:, :, 0] - base[:, :, 0])) < 1e-5
    assert np.max(np.abs(pert[:, :, 3] - base[:, :, 3])) > 1e-4
    # zero query: uniform weights, so the mean of the decoded values
    z = _lut_run(np.zeros_like(q[:, :, :1]), ki, kcb, vi, vcb, scale)
    np.testing.assert_allclose(z[0, 0, 0], ov.dequantize_vq(vi, vcb)[0, 0].mean(0), atol=1e-5)
    # large logits: a softmax that does not overflow
    big = _lut_run(q * 40, ki, kcb, vi, vcb, 1.0)
    ref = ov.fused_sdpa(q * 40, ki, kcb, vi, vcb, 1.0)
    assert np.isfinite(big).all() and np.max(np.abs(big - ref)) < LUT_TOL


def test_lut_attention_errors():
    """messages of veloxquant_mlx/metal/fused_sdpa.py:229-248 plus this kernel's own limits"""
    require_gpu()
    q, ki, kcb, vi, vcb = _lut_case(1, 4, 4, 1, 32, 64, 4, 4, 256, seed=1)
    t = lambda *xs: [to_dev(x) for x in xs]
    with pytest.raises(ValueError, match="must equal n_sub"):
        K.metal_fused_sdpa(*t(q[..., :60], ki, kcb, vi, vcb), 0.1)
    with pytest.raises(ValueError, match="same n_centroids"):
        K.metal_fused_sdpa(*t(q, ki, kcb, vi, vcb[:128]), 0.1)
    with pytest.raises(ValueError, match="multiple of H_kv"):
        K.metal_fused_sdpa(*t(np.concatenate([q, q[:, :1]], 1), ki, kcb, vi, vcb), 0.1)
    big = np.random.default_rng(0).standard_normal((512, 4)).astype(np.float32)
    with pytest.raises(ValueError, match="exceeds 256"):
        K.metal_fused_sdpa(*t(q, ki.astype(np.int32), big, vi.astype(np.int32), big), 0.1)
    with pytest.raises(ValueError, match="S_q"):
        K.metal_fused_sdpa(*t(np.repeat(q, 40, 2), ki, kcb, vi, vcb), 0.1, causal=True)
    with pytest.raises(RuntimeError, match="ROCm device"):
        K.metal_fused_sdpa(torch.from_numpy(q), *t(ki, kcb, vi, vcb), 0.1)


def test_lut_attention_many_weights_below_one_unit_still_count():
    """One dominant token and thousands whose weights are each below the resolution of the
    integer histogram (2^-18 of the largest weight in blocks of 8192 tokens): their total is a
    few percent of the sum and must not be rounded away."""
    require_gpu()
    rng = np.random.default_rng(3)
    B, H, S, D, sub, C = 16, 8, 8192, 64, 4, 256
    kcb = (rng.standard_normal((C, sub)) * 0.05).astype(np.float32)
    kcb[7] = [3.0, -3.0, 3.0, -3.0]
    vcb = rng.standard_normal((C, sub)).astype(np.float32)
    ki = rng.integers(8, C, (B, H, S, D // sub)).astype(np.uint8)
    vi = rng.integers(0, C, (B, H, S, D // sub)).astype(np.uint8)
    ki[:, :, 100] = 7
    q = np.tile(kcb[7], D // sub)[None, None, None, :].repeat(B, 0).repeat(H, 1).astype(np.float32)
    # the dominant score is 16 * 36 * scale, the others are near zero: a gap of about 13.5 nats
    scale = 13.5 / (16 * 36)
    ref = ov.fused_sdpa(q, ki, kcb, vi, vcb, scale)
    w_small = np.exp(-13.5) * (S - 1)
    assert 0.005 < w_small < 0.05 and np.exp(-13.5) * 2 ** 18 < 0.5
    got = _lut_run(q, ki, kcb, vi, vcb, scale)
    dom = ov.dequantize_vq(vi, vcb)[:, :, 100:101]
    assert np.max(np.abs(ref - dom)) > 5e-3          # the small weights matter at the tolerance below
    assert np.max(np.abs(got - ref)) < 2e-4


# ---------------------------------------------------------------------------
# fused key encode (+ decode): smooth, Walsh-Hadamard transform, assignment, way back
# ---------------------------------------------------------------------------

def _gap_to_second(k_tilde, cb, sub):
    """relative gap between the two smallest squared distances of every sub-vector"""
    x = k_tilde.reshape(-1, sub).astype(np.float64)
    d = ((x[:, None, :] - cb[None].astype(np.float64)) ** 2).sum(-1)
    d.sort(axis=1)
    return ((d[:, 1] - d[:, 0]) / np.maximum(d[:, 1], 1e-30)).reshape(k_tilde.shape[:-1] + (-1,))


@pytest.mark.parametrize("D,sub", [(64, 8), (128, 8), (256, 8), (512, 8), (32, 4), (64, 4), (128, 4), (256, 4)])
def test_encode_keys_on_integer_keys_is_exact(D, sub):
    """Integer keys and power-of-two smoothing factors: every partial sum of the transform is
    exact in float32 whatever its order, so the transformed keys, hence the indices, must equal
    the oracle's bit for bit."""
    require_gpu()
    rng = np.random.default_rng(D + sub)
    B, Hh, S, C = 2, 3, 21, 200
    keys = rng.integers(-8, 9, (B, Hh, S, D)).astype(np.float16)
    smooth = (2.0 ** rng.integers(-2, 3, (Hh, D))).astype(np.float32)
    Hm = ov.walsh_hadamard_matrix(D)
    cb = rng.standard_normal((C, sub)).astype(np.float32)
    kt_ref, idx_ref, khat_ref = ov.encode_decode_keys(keys, smooth, Hm, cb, sub)
    k_hat, idx, k_tilde = K.vecinfer_encode_decode_metal(to_dev(keys), to_dev(cb), sub, to_dev(Hm), to_dev(smooth),
                                                          want_k_tilde=True)
    np.testing.assert_array_equal(host(k_tilde), kt_ref)
    np.testing.assert_array_equal(host(idx), idx_ref)
    assert k_hat.dtype == torch.float16 and k_hat.shape == keys.shape
    np.testing.assert_allclose(host(k_hat).astype(np.float32), khat_ref, rtol=1.5e-3, atol=1e-3)
    # indices only, one byte each
    none, idx8 = K.vecinfer_encode_decode_metal(to_dev(keys), to_dev(cb), sub, to_dev(Hm), to_dev(smooth),
                                                index_dtype=torch.uint8, want_k_hat=False)
    assert none is None
    np.testing.assert_array_equal(host(idx8), idx_ref.astype(np.uint8))


# the forms for more than 512 centroids: SPLIT up to 32768 sub-vectors against more than 1024 centroids (three heads: on both sides
# of that), the image of the whole codebook otherwise; one lane group of a token each way
@pytest.mark.parametrize("D,sub,nc,S", [
    (128, 4, 4096, 1), (128, 4, 4096, 341), (128, 4, 4096, 342), (64, 4, 4096, 682), (64, 4, 4096, 683), (256, 4, 4096, 170), (256, 4, 4096, 171),
    (128, 8, 2048, 682), (128, 8, 2048, 683), (512, 8, 2048, 20), (64, 8, 1500, 3), (32, 4, 1100, 77), (128, 4, 1000, 50), (256, 8, 600, 33),
])
@pytest.mark.parametrize("smooth_rows", [None, "vector", "heads"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, "integers"])
def test_encode_keys_with_large_codebooks(dtype, smooth_rows, D, sub, nc, S):
    """Indices exact on the kernel's own transformed keys; those exact on integer keys, and elsewhere no further from float64
    than the float32 product that they replace; the way back from the kernel's own indices."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(D + nc + S)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    whole = dtype == "integers"
    keys = torch.randint(-8, 9, (1, 3, S, D), generator=gen, device="cuda").half() if whole else (r(1, 3, S, D) * r(D).exp()).to(dtype)
    shape = {None: None, "vector": (D,), "heads": (3, D)}[smooth_rows]
    smooth = None if shape is None else torch.exp2(torch.randint(-2, 3, shape, generator=gen, device="cuda").float()) if whole else r(*shape).exp()
    Hm, cb = to_dev(ov.walsh_hadamard_matrix(D)), r(nc, sub) * D ** 0.25
    k_hat, idx, k_tilde = K.vecinfer_encode_decode_metal(keys, cb, sub, Hm, smooth, want_k_tilde=True)
    wide = lambda t: 1.0 if t is None else t[:, None, :] if t.ndim == 2 else t
    exact = (keys.double() / wide(None if smooth is None else smooth.double())) @ Hm.double()
    product = (keys.float() / wide(smooth)) @ Hm
    err = lambda t: float((t.double() - exact).norm() / exact.norm())
    if whole:   # every partial sum is a whole number of quarters below 2^24: only the last step, times the matrix' magnitude, rounds
        h = float(Hm[0, 0])
        assert torch.equal(k_tilde, ((keys.double() / wide(None if smooth is None else smooth.double())) @ (Hm.double() / h)).float() * h)
    assert err(k_tilde) <= 1.05 * max(err(product), 2.0 ** -25)
    np.testing.assert_array_equal(host(idx).reshape(-1), cref.vq_assign(host(k_tilde).reshape(-1, sub), host(cb), sub).reshape(-1))
    back = (cb.double()[idx.long()].reshape(exact.shape) @ Hm.double()) * wide(None if smooth is None else smooth.double())
    # log2(D) + 2 roundings of 2^-24 of the row's own size, and the output type's
    tol = 2.0 ** -11 if keys.dtype == torch.float16 else 0.0
    row = back.norm(dim=-1, keepdim=True) * (1 if smooth is None else float(smooth.max() / smooth.min()))
    assert ((k_hat.double() - back).abs() <= back.abs() * tol + row * 2.0 ** -24 * (D.bit_length() + 2) + 6e-8).all()


def test_encode_keys_at_any_storage_offset():
    """Keys and smoothing factors that are contiguous but start between 16-byte boundaries, at codebooks on both sides of 256
    centroids: the same values as from aligned memory."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    keys, smooth, Hm = r(1, 2, 7, 128).half(), r(2, 128).exp(), to_dev(ov.walsh_hadamard_matrix(128))
    moved = torch.empty(keys.numel() + 1, dtype=keys.dtype, device="cuda")[1:].view(keys.shape).copy_(keys)
    smooth_moved = torch.empty(smooth.numel() + 3, device="cuda")[3:].view(smooth.shape).copy_(smooth)
    assert moved.is_contiguous() and moved.data_ptr() % 16 and smooth_moved.data_ptr() % 16
    for nc, sub in ((4096, 4), (2048, 8), (256, 8)):
        cb = r(nc, sub)
        ref = K.vecinfer_encode_decode_metal(keys, cb, sub, Hm, smooth, want_k_tilde=True)
        for k, sm in ((moved, smooth), (keys, smooth_moved)):
            assert all(torch.equal(a, b) for a, b in zip(K.vecinfer_encode_decode_metal(k, cb, sub, Hm, sm, want_k_tilde=True), ref))


def test_encode_keys_with_a_large_codebook_keeps_the_gradient_of_the_factors():
    """Above 256 centroids the reconstruction (centroids @ H^T) * smooth carries gradients to the smoothing factors, and the
    transformed keys to the keys."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(6)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    keys, smooth, cb, Hm = r(1, 2, 9, 64), r(2, 64).exp(), r(1024, 4), to_dev(ov.walsh_hadamard_matrix(64))
    sm, kk = smooth.clone().requires_grad_(), keys.clone().requires_grad_()
    k_hat, _, k_tilde = K.vecinfer_encode_decode_metal(keys, cb, 4, Hm, sm, want_k_tilde=True)
    g, = torch.autograd.grad(k_hat.sum(), sm)
    torch.testing.assert_close(g, (k_hat.detach() / smooth[None, :, None]).sum(dim=(0, 2)), rtol=1e-4, atol=1e-3)
    *_, k_tilde = K.vecinfer_encode_decode_metal(kk, cb, 4, Hm, smooth, want_k_tilde=True)
    g, = torch.autograd.grad(k_tilde.sum(), kk)
    torch.testing.assert_close(g, (Hm.sum(1) / smooth[:, None])[None].expand_as(g), rtol=1e-4, atol=1e-4)
    with torch.no_grad():   # nothing to differentiate: the fused launch, at the same values
        k_fused, _ = K.vecinfer_encode_decode_metal(keys, cb, 4, Hm, sm)
    torch.testing.assert_close(k_fused, k_hat.detach(), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("smooth_rows", [None, 1, "heads", "vector"])
def test_encode_keys_random_keys(dtype, smooth_rows):
    require_gpu()
    rng = np.random.default_rng(11)
    B, Hh, S, D, sub, C = 2, 4, 333, 128, 8, 256
    keys_t = to_dev((rng.standard_normal((B, Hh, S, D)) * np.exp(rng.standard_normal(D))).astype(np.float32), dtype)
    keys = host(keys_t).astype(np.float32)
    smooth = {None: None, 1: np.exp(rng.standard_normal((1, D)) * 0.5), "heads": np.exp(rng.standard_normal((Hh, D)) * 0.5),
              "vector": np.exp(rng.standard_normal(D) * 0.5)}[smooth_rows]
    smooth = None if smooth is None else smooth.astype(np.float32)
    Hm = ov.walsh_hadamard_matrix(D)
    cb = rng.standard_normal((C, sub)).astype(np.float32)
    kt_ref, idx_ref, _ = ov.encode_decode_keys(keys, smooth, Hm, cb, sub)
    k_hat, idx, k_tilde = K.vecinfer_encode_decode_metal(keys_t, to_dev(cb), sub, to_dev(Hm),
                                                          None if smooth is None else to_dev(smooth), want_k_tilde=True)
    kt, idx = host(k_tilde), host(idx)
    # the transform: float32 butterflies against the float64 product
    assert np.max(np.abs(kt - kt_ref)) <= 2e-6 * np.max(np.abs(kt_ref))
    # the assignment is exact on the kernel's own transformed keys
    np.testing.assert_array_equal(idx, ov.quantize_vq(kt, cb, sub))
    # against the oracle's transformed keys only near ties may differ
    diff = idx != idx_ref
    assert diff.mean() < 1e-3
    if diff.any():
        assert _gap_to_second(kt_ref, cb, sub)[diff].max() < 1e-4
    # the way back, from the kernel's own indices
    sm = 1.0 if smooth is None else (smooth[:, None, :] if smooth.ndim == 2 and smooth.shape[0] == Hh else smooth.reshape(-1, D)[0])
    back = (ov.dequantize_vq(idx, cb).astype(np.float64) @ Hm.T.astype(np.float64)) * sm
    tol = {torch.float16: 1.5e-3, torch.bfloat16: 1e-2, torch.float32: 1e-5}[dtype]
    assert k_hat.dtype == dtype
    np.testing.assert_allclose(host(k_hat).astype(np.float64), back, rtol=tol, atol=tol)


def test_encode_keys_other_shapes_take_the_composition():
    """sub_dim 16, a non-Hadamard matrix, a codebook past what a block holds: same contract through the
    matrix product and the assignment / gather kernels."""
    require_gpu()
    rng = np.random.default_rng(2)
    keys = rng.standard_normal((1, 2, 40, 64)).astype(np.float16)
    Hm = ov.walsh_hadamard_matrix(64)
    for sub, C, Hmat in ((16, 64, Hm), (8, 2100, Hm), (8, 64, np.linalg.qr(rng.standard_normal((64, 64)))[0].astype(np.float32))):
        cb = rng.standard_normal((C, sub)).astype(np.float32)
        k_hat, idx, k_tilde = K.vecinfer_encode_decode_metal(to_dev(keys), to_dev(cb), sub, to_dev(Hmat), want_k_tilde=True)
        np.testing.assert_array_equal(host(idx), ov.quantize_vq(host(k_tilde), cb, sub))
        np.testing.assert_allclose(host(k_tilde), keys.astype(np.float32) @ Hmat, rtol=1e-4, atol=1e-4)
        back = ov.dequantize_vq(host(idx), cb) @ Hmat.T
        np.testing.assert_allclose(host(k_hat).astype(np.float32), back, rtol=2e-3, atol=2e-3)
    v_hat, v_idx = K.vecinfer_encode_decode_simple_metal(to_dev(keys), to_dev(cb), 8)
    np.testing.assert_array_equal(host(v_idx), ov.quantize_vq(keys, cb, 8))
    np.testing.assert_allclose(host(v_hat).astype(np.float32), ov.dequantize_vq(host(v_idx), cb), rtol=1e-3, atol=1e-3)
    with pytest.raises(ValueError, match="must be 4D"):
        K.vecinfer_encode_decode_metal(to_dev(keys[0]), to_dev(cb), 8, to_dev(Hm))
    with pytest.raises(ValueError, match="not divisible"):
        K.vecinfer_encode_decode_metal(to_dev(keys), to_dev(cb), 7, to_dev(Hm))


@pytest.mark.parametrize("modes", [{}, dict(fused_sdpa=True), dict(fused_sdpa=True, fused_sdpa_memory_bound=True)])
@pytest.mark.parametrize("key_bits,key_sub", [(12, 4), (8, 8), (4, 16)])
def test_cache_under_inference_mode(modes, key_bits, key_sub):
    """Filled and attended under ``torch.inference_mode``, from its first keys on and from a restored state on: the values of a
    cache outside of it."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(8)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    cfg = KVCacheConfig(method="vecinfer", head_dim=64, key_codebook_bits=key_bits, key_sub_dim=key_sub, smooth_factors=r(2, 64).exp(),
                        key_codebook=r(1 << key_bits, key_sub), value_codebook=r(256, 8), **modes)
    k, v, q = r(1, 2, 70, 64).half(), r(1, 2, 70, 64).half(), r(1, 4, 1, 64).half()

    def use():
        c = KVCacheFactory.create(cfg)
        outs = [*c.update_and_fetch(k, v), *c.update_and_fetch(k[:, :, :1], v[:, :, :1])]
        if modes:
            outs.append(c.fused_sdpa(q, 0.1))
            d = KVCacheFactory.create(cfg)
            d.state = c.state
            outs += [d.fused_sdpa(q, 0.1), d.fused_sdpa(q, 0.1)]
        return outs
    want = use()
    with torch.inference_mode():
        got = use()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("B,Hq,Hkv,D,S,n,sub,by_index", [
    (1, 4, 1, 128, 1, 3000, 8, True), (48, 32, 8, 128, 1, 1537, 8, False), (32, 8, 8, 128, 1, 3072, 8, True), (32, 8, 8, 128, 1, 3073, 8, False),
    (32, 8, 8, 64, 1, 4096, 8, True), (32, 8, 8, 64, 1, 4097, 8, False), (16, 16, 8, 128, 4, 3073, 8, False), (32, 8, 8, 128, 1, 3073, 4, True),
    (64, 4, 4, 256, 1, 1537, 8, False), (64, 4, 4, 256, 1, 1536, 8, True), (1, 4, 1, 128, 9, 40, 8, False),
])
def test_few_rows_over_small_codebooks_take_the_kernel_of_their_depth(monkeypatch, B, Hq, Hkv, D, S, n, sub, by_index):
    """Both sides of the rule between the index kernel and the table kernel, which agree."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(n)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    cfg = KVCacheConfig(method="vecinfer", head_dim=D, key_codebook_bits=8, key_sub_dim=sub, key_codebook=r(256, sub),
                        value_codebook=r(256, 8), fused_sdpa=True, fused_sdpa_memory_bound=True)
    c = KVCacheFactory.create(cfg)
    idx = lambda s: torch.randint(0, 256, (B, Hkv, n, D // s), generator=gen, device="cuda", dtype=torch.uint8)
    c.state, q = (idx(sub), idx(8)), r(B, Hq, S, D)
    real, calls = K.vecinfer_attend_indices, []

    def spy(*a, **k):
        calls.append(real(*a, **k))
        return calls[-1]
    monkeypatch.setattr(K, "vecinfer_attend_indices", spy)
    out = c.fused_sdpa(q, 0.1 / D ** 0.5)
    assert (len(calls) == 1 and calls[0] is not None) == by_index
    monkeypatch.setattr(K, "vecinfer_attend_indices", (lambda *a, **k: None) if by_index else real)
    kw = dict(n_tokens=n, H_mat=c._H, causal=S > 1)
    other = c.fused_sdpa(q, 0.1 / D ** 0.5) if by_index else real(q, *c.state[:1], c._key_codebook, c.state[1], c._value_codebook, 0.1 / D ** 0.5, **kw)
    # both sum in float32 over at most 4097 tokens of unit variance; scores of a few units, D of them rounded
    assert other is None or float((out - other).abs().max()) < 2e-4


def test_matrix_made_inside_a_graph_is_not_kept_for_eager_calls():
    """A restored cache whose first call is captured: the matrix of that capture holds nothing until a replay, so a call outside
    makes its own, and the graph replays to the same values."""
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(12)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")
    cfg = KVCacheConfig(method="vecinfer", head_dim=64, key_codebook_bits=4, key_sub_dim=16, key_codebook=r(16, 16), value_codebook=r(256, 8),
                        smooth_factors=r(2, 64).exp(), fused_sdpa=True, fused_sdpa_memory_bound=True)
    a, b, q = KVCacheFactory.create(cfg), KVCacheFactory.create(cfg), r(1, 4, 1, 64)
    a.update_and_fetch(r(1, 2, 90, 64), r(1, 2, 90, 64))
    want = a.fused_sdpa(q, 0.1)
    b.state = a.state
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = b.fused_sdpa(q, 0.1)
    assert torch.equal(b.fused_sdpa(q, 0.1), want)
    for _ in range(3):
        graph.replay()
        assert torch.equal(out, want) and torch.equal(b.fused_sdpa(q, 0.1), want)


@pytest.mark.parametrize("B,H,S,D,kn,ks,vn,vs,dtype,rows", [
    (2, 8, 1, 128, 4096, 4, 256, 8, torch.float16, 8), (1, 3, 5, 64, 256, 8, 256, 8, torch.bfloat16, 1), (1, 4, 1, 256, 4096, 4, 2048, 8, torch.float32, 0),
    (4, 8, 3, 128, 33, 4, 4096, 4, torch.float16, 1), (1, 1, 1, 512, 2048, 8, 7, 8, torch.bfloat16, 0), (8, 8, 5, 128, 300, 4, 31, 8, torch.float16, 8),
    (1, 16, 21, 128, 256, 8, 256, 8, torch.float16, 1), (5, 2, 1, 32, 1, 4, 1, 8, torch.float32, 2), (8, 8, 6, 128, 256, 4, 256, 8, torch.float16, 1)])
def test_step_indices_go_into_the_store(B, H, S, D, kn, ks, vn, vs, dtype, rows):
    """A few tokens in one launch, into the store at a token of its own, against the two launches with the same rule: the
    same whole numbers, and nothing else of the store touched.  The last row is more than one round of blocks takes
    and must be refused."""
    require_gpu()
    g = torch.Generator(device="cuda").manual_seed(B * D + S + kn)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")
    keys, values = (rand(B, H, S, D) * torch.exp(rand(D))).to(dtype), rand(B, H, S, D).to(dtype)
    keys[0, 0, 0, :ks] = 300.0 if S > 1 else 0.0
    kcb, vcb = rand(kn, ks), rand(vn, vs)
    smooth = None if rows == 0 else torch.exp(0.3 * rand(rows, D))
    Hm = walsh_hadamard_matrix(D, device="cuda")
    it = lambda n: torch.uint8 if n <= 256 else torch.int32
    cap, at = S + 9, 5
    ks_store = torch.full((B, H, cap, D // ks), 77, dtype=it(kn), device="cuda")
    vs_store = torch.full((B, H, cap, D // vs), 77, dtype=it(vn), device="cuda")
    want_k, want_v = ks_store.clone(), vs_store.clone()
    took = K.vecinfer_encode_step(keys, values, kcb, ks, vcb, vs, Hm, smooth, ks_store, vs_store, at)
    assert took == (-(-B * H * S * D // ks // 64) + -(-B * H * S * D // vs // 64) <= 256)
    if took:
        want_k[:, :, at:at + S] = K.vecinfer_encode_decode_metal(keys, kcb, ks, Hm, smooth, index_dtype=it(kn), want_k_hat=False)[1]
        want_v[:, :, at:at + S] = K.vecinfer_quantize_metal(values, vcb, vs, index_dtype=it(vn))
    assert torch.equal(ks_store, want_k) and torch.equal(vs_store, want_v)
    # what does not fit the store is refused by the library before any launch
    assert not K.vecinfer_encode_step(keys, values, kcb, ks, vcb, vs, Hm, smooth, ks_store, vs_store, cap - S + 1)
    assert torch.equal(ks_store, want_k) and torch.equal(vs_store, want_v)


def test_factors_of_another_width_are_refused():
    """Smoothing factors whose rows are not as wide as a head: not taken by the step's launch, refused by the cache at the update
    and by the fused encode, and nothing stored."""
    require_gpu()
    r = lambda *s: torch.randn(s, device="cuda")
    B, H, D = 1, 4, 128
    keys, values, kcb, vcb = r(B, H, 1, D).half(), r(B, H, 1, D).half(), r(256, 8), r(256, 8)
    Hm = walsh_hadamard_matrix(D, device="cuda")
    stores = [torch.full((B, H, 4, D // 8), 77, dtype=torch.uint8, device="cuda") for _ in range(2)]
    for smooth in (r(64).exp(), r(H, 64).exp(), r(1, 96).exp(), r(1, 1, D).exp(), torch.ones((), device="cuda")):
        assert not K.vecinfer_encode_step(keys, values, kcb, 8, vcb, 8, Hm, smooth, *stores, 1)
    assert all(bool((s == 77).all()) for s in stores)
    for smooth in (r(64).exp(), r(H, 64).exp()):
        with pytest.raises(RuntimeError):
            K.vecinfer_encode_decode_metal(keys, kcb, 8, Hm, smooth)
        c = KVCacheFactory.create(KVCacheConfig(method="vecinfer", head_dim=D, key_codebook_bits=8, key_sub_dim=8, key_codebook=kcb, value_codebook=vcb,
                                                smooth_factors=smooth, fused_sdpa=True, fused_sdpa_memory_bound=True))
        with pytest.raises(RuntimeError):
            c.update_and_fetch(keys, values)
        assert c.offset == 0 and c._stored_S_kv == 0


@pytest.mark.parametrize("nc", [1, 3, 16, 17, 31, 32, 33, 64])
@pytest.mark.parametrize("odd", ["plain", "nan", "all nan", "inf", "equal"])
def test_step_over_codebooks_of_a_tile_or_two(nc, odd):
    """A codebook of one tile, whose two cells are all there is, and the first of two: the indices of the two launches, with
    centroids and sub-vectors that are no numbers, infinite ones and equal ones."""
    require_gpu()
    g = torch.Generator(device="cuda").manual_seed(nc)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")
    B, H, D = 3, 4, 128
    keys, values = rand(B, H, 1, D).half(), rand(B, H, 1, D).half()
    values[0, 0, 0, 5], values[0, 1, 0, 17], values[0, 2, 0] = float("nan"), float("inf"), 0.0
    kcb, vcb = rand(nc, 4), rand(nc, 8)
    for cb in (kcb, vcb):
        if odd == "nan":
            cb[nc // 2, 1] = float("nan")
        elif odd == "all nan":
            cb[:] = float("nan")
        elif odd == "inf":
            cb[nc - 1, 0] = float("inf")
        elif odd == "equal":
            cb[:] = cb[0].clone()
    Hm = walsh_hadamard_matrix(D, device="cuda")
    ks, vs = (torch.full((B, H, 2, D // n), 99, dtype=torch.uint8, device="cuda") for n in (4, 8))
    assert K.vecinfer_encode_step(keys, values, kcb, 4, vcb, 8, Hm, None, ks, vs, 1)
    assert torch.equal(ks[:, :, 1:], K.vecinfer_encode_decode_metal(keys, kcb, 4, Hm, index_dtype=torch.uint8, want_k_hat=False)[1])
    assert torch.equal(vs[:, :, 1:], K.vecinfer_quantize_metal(values, vcb, 8, index_dtype=torch.uint8))
