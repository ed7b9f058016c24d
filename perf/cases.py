"""Performance cases of the KV-cache compression path on one GPU.

Every case is work that a program serving a language model has this package do, through the cache classes
or the kernel functions it would call itself:

* ``step``    two decode steps of one layer: ``update_and_fetch`` of one token a sequence, then ``fused_sdpa``
  over the packed KIVI cache (2 / 3 / 4 bits, heads of 64 / 128 / 256 channels, ragged batches)
* ``stack``   two decode steps of all layers of a model whose caches share one stack (one launch for all layers)
* ``prefill`` a whole prompt, chunk by chunk, into an empty packed cache, attending causally after every chunk
* ``flash``   causal self-attention over plain keys and values
* ``scalar``  the kernel function over uint8 codes and float32 scale / zero (one query token a sequence)
* ``vecstep`` two decode steps over a VecInfer cache that holds codebook indices only
* ``fill``    a prompt handed to one of the caches that return reconstructed keys and values

Head shapes are those of the models the package is used with (query heads, kv heads, head size).  Keys are
N(0,1) with log-normal factors a channel (outlier channels), values and queries N(0,1).

The decode passes take two steps and then drop both tokens again (``trim``, what a speculative decoder does with
rejected tokens), so that a pass can be repeated and its second output shows that its first token was stored.
"""

from __future__ import annotations

import math

import torch

from veloxquant_mlx_amd import kernels as K
from veloxquant_mlx_amd.allocators.vecinfer import (apply_dual_transform_keys, calibrate_smooth_factors,
                                                    walsh_hadamard_matrix)
from veloxquant_mlx_amd.cache import KVCacheConfig, KVCacheFactory, LayerStackedKIVICache

RESIDUAL = 128   # newest tokens kept exact, the caches' default
STEPS = 2        # decode steps of a pass
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
HEADS = [(32, 8, 128), (24, 8, 128), (28, 4, 128), (40, 10, 128), (32, 8, 64), (14, 2, 64), (9, 3, 64), (12, 4, 256), (8, 4, 256)]
CHUNK = 4096     # tokens made and stored at a time while a long context is set up


def listed():
    return [
        # a short chat on a small model's default settings: launch latency and host work are all there is
        dict(name="step_short", kind="step", hq=32, hkv=8, d=64, batch=1, ctx=700, bits=2, group=32, dtype="float16", ragged=False),
        # one user, 8k tokens of context, 2 bits
        dict(name="step_8k", kind="step", hq=32, hkv=8, d=128, batch=1, ctx=8320, bits=2, group=32, dtype="float16", ragged=False),
        # a serving batch at 32k, 4 bits: the bytes of the cache count
        dict(name="step_32k_batch", kind="step", hq=32, hkv=8, d=128, batch=16, ctx=32900, bits=4, group=64, dtype="float16", ragged=False),
        # heads of 256 channels, a right-padded batch of an odd size whose sequences differ in length
        dict(name="step_d256_ragged", kind="step", hq=12, hkv=4, d=256, batch=7, ctx=20011, bits=2, group=32, dtype="bfloat16", ragged=True),
        # all 36 layers of a model at 32k in one launch: the largest
        dict(name="stack_36", kind="stack", hq=32, hkv=8, d=128, layers=36, batch=8, ctx=32900, bits=4, group=64, dtype="float16"),
        # a long prompt in chunks of 512, quantised as it is written
        dict(name="prefill_8k", kind="prefill", hq=32, hkv=8, d=128, batch=1, tokens=8192, chunk=512, bits=4, group=32, dtype="bfloat16"),
        # self-attention of a whole prompt over plain fp16 keys and values
        dict(name="flash_4k", kind="flash", hq=32, hkv=32, d=128, batch=1, tokens=4096),
        # the kernel function over byte codes: 4-bit levels, one query token
        dict(name="scalar_8k", kind="scalar", hq=32, hkv=8, d=128, batch=2, tokens=8192, bits=4, group=32),
        # VecInfer's default codebooks (4096 x 4 keys, 256 x 8 values), a small batch with an odd context
        dict(name="vecstep_default", kind="vecstep", hq=32, hkv=8, d=128, batch=2, ctx=9001, key_bits=12, key_sub=4, dtype="float16"),
        # a prompt into the default KIVI cache
        dict(name="fill_kivi", kind="fill", method="kivi", hkv=8, d=128, batch=1, tokens=2048, dtype="float16"),
        # a batch of prompts into the sliding-window cache with clip search and channel reordering
        dict(name="fill_skvq", kind="fill", method="skvq", hkv=8, d=128, batch=8, tokens=4100, dtype="float16"),
        # a prompt encoded with VecInfer's default codebooks
        dict(name="fill_vecinfer", kind="fill", method="vecinfer", hkv=8, d=128, batch=1, tokens=4096, dtype="float16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fits(tokens, most):
    return max(1, min(tokens, most))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "stack", "prefill", "prefill", "flash", "scalar", "vecstep", "fill", "fill", "fill"])
    hq, hkv, d = rng.choice(HEADS)
    dtype = rng.choice(["float16", "float16", "bfloat16"])
    bits, group = rng.choice([(2, 32), (2, 32), (4, 32), (4, 64), (3, 32)])
    if kind == "step":
        batch = _log_int(rng, 1, 16)
        ctx = _fits(_log_int(rng, 400, 33000), (16 * 32768 * 8 * 128) // (batch * hkv * d))
        return dict(kind=kind, hq=hq, hkv=hkv, d=d, batch=batch, ctx=ctx, bits=bits, group=group, dtype=dtype,
                    ragged=batch > 1 and rng.random() < 0.3)
    if kind == "stack":
        hq, hkv, d = rng.choice([h for h in HEADS if h[2] == 128])
        layers, batch = rng.choice([16, 24, 28, 32, 36]), _log_int(rng, 1, 8)
        ctx = _fits(_log_int(rng, 1000, 33000), (36 * 8 * 32768 * 8 * 128) // (layers * batch * hkv * d))
        return dict(kind=kind, hq=hq, hkv=hkv, d=d, layers=layers, batch=batch, ctx=ctx, bits=bits, group=group, dtype=dtype)
    if kind == "prefill":
        return dict(kind=kind, hq=hq, hkv=hkv, d=d, batch=rng.choice([1, 1, 2]), tokens=_log_int(rng, 600, 6000),
                    chunk=rng.choice([256, 512, 512, 1024, 2048]), bits=bits, group=group, dtype=dtype)
    if kind == "flash":
        hkv = rng.choice([hkv, hq])
        return dict(kind=kind, hq=hq, hkv=hkv, d=d, batch=rng.choice([1, 1, 2]), tokens=_log_int(rng, 400, 5000 if d < 256 else 2500))
    if kind == "scalar":
        batch = _log_int(rng, 1, 4)
        return dict(kind=kind, hq=hq, hkv=hkv, d=d, batch=batch, tokens=_log_int(rng, 500, 16384), bits=rng.choice([2, 4, 4, 8]), group=32)
    if kind == "vecstep":
        hq, hkv, d = rng.choice([(32, 8, 128), (24, 8, 128), (28, 4, 128), (32, 8, 64), (12, 4, 256)])
        key_bits, key_sub = rng.choice([(12, 4), (12, 4), (8, 8)])
        return dict(kind=kind, hq=hq, hkv=hkv, d=d, batch=_log_int(rng, 1, 4), ctx=_log_int(rng, 400, 16384), key_bits=key_bits,
                    key_sub=key_sub, dtype=dtype)
    method = rng.choice(["kivi", "kivi", "kitty", "age_tiered", "skvq", "zipcache", "vecinfer"])
    batch = _log_int(rng, 1, 8)
    return dict(kind="fill", method=method, hkv=hkv, d=d, batch=batch, tokens=_fits(_log_int(rng, 300, 8192), 8 * 4100 * 8 * 128 // (batch * hkv * d)),
                dtype=dtype)


# ---------------------------------------------------------------------------
# inputs and objects a user's program has in hand before the call
# ---------------------------------------------------------------------------

class _Source:
    """Keys, values and queries made on the GPU from a seed."""

    def __init__(self, seed, d):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.factors = torch.exp(self.normal(d))

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def keys(self, dtype, *shape):
        return (self.normal(*shape) * self.factors).to(dtype)

    def values(self, dtype, *shape):
        return self.normal(*shape).to(dtype)


def _kivi_config(case, **more):
    return KVCacheConfig(method="kivi", head_dim=case["d"], bit_width_inlier=case["bits"], kivi_group_size=case["group"],
                         residual_length=RESIDUAL, fused_sdpa=True, fused_sdpa_memory_bound=True, **more)


def _fill_context(cache, src, case, ctx):
    dtype = DTYPES[case["dtype"]]
    for at in range(0, ctx, CHUNK):
        shape = (case["batch"], case["hkv"], min(CHUNK, ctx - at), case["d"])
        cache.update_and_fetch(src.keys(dtype, *shape), src.values(dtype, *shape))


def _between_flushes(ctx, group):
    """``ctx`` or a little less: a context to which ``STEPS`` tokens can be appended without a flush."""
    return ctx - max(0, (ctx - RESIDUAL) % group + STEPS + 1 - group)


def _new_tokens(src, case, dtype, *lead):
    """Keys, values and queries of the tokens of a pass, layer by layer where there are several."""
    kv, q = (*lead, case["batch"], case["hkv"], 1, case["d"]), (*lead, case["batch"], case["hq"], 1, case["d"])
    return [(src.keys(dtype, *kv), src.values(dtype, *kv), src.values(dtype, *q)) for _ in range(STEPS)]


def prepare(case, seed):
    src = _Source(seed, case["d"])
    kind, d, batch, hkv = case["kind"], case["d"], case["batch"], case["hkv"]
    st = {"case": case, "scale": 1.0 / math.sqrt(d)}
    if kind in ("step", "stack"):
        dtype, ctx = DTYPES[case["dtype"]], _between_flushes(case["ctx"], case["group"])
        layers = case["layers"] if kind == "stack" else 1
        cfg = _kivi_config(case, fused_sdpa_max_ctx=-(-(ctx + 256) // 256) * 256)
        if kind == "stack":
            cache = LayerStackedKIVICache(cfg, layers)
            for l in range(layers):
                _fill_context(cache[l], src, case, ctx)
            # the stack a generation in progress has: its layers' buffers are slices of one
            cache.fused_sdpa_all(src.values(dtype, layers, batch, case["hq"], 1, d), st["scale"])
        else:
            cache = KVCacheFactory.create(cfg)
            _fill_context(cache, src, case, ctx)
        lead = (layers,) if kind == "stack" else ()
        lengths = [None] * STEPS
        if case.get("ragged"):
            low = max(1, ctx // 3)
            first = low + torch.randint(0, ctx + 1 - low, (batch,), generator=src.gen, device="cuda")
            lengths = [first + 1 + t for t in range(STEPS)]
        st.update(cache=cache, lengths=lengths, tokens=_new_tokens(src, case, dtype, *lead))
    elif kind == "prefill":
        dtype, n = DTYPES[case["dtype"]], case["tokens"]
        chunks = []
        for at in range(0, n, case["chunk"]):
            m = min(case["chunk"], n - at)
            chunks.append((src.keys(dtype, batch, hkv, m, d), src.values(dtype, batch, hkv, m, d), src.values(dtype, batch, case["hq"], m, d)))
        st.update(chunks=chunks, config=_kivi_config(case, fused_sdpa_max_ctx=-(-n // 64) * 64))
    elif kind == "flash":
        n = case["tokens"]
        st.update(q=src.values(torch.float16, batch, case["hq"], n, d), k=src.values(torch.float16, batch, hkv, n, d),
                  v=src.values(torch.float16, batch, hkv, n, d))
    elif kind == "scalar":
        n, levels = case["tokens"], (1 << case["bits"]) - 1
        kq = K.kivi_quant_codes(src.keys(torch.float16, batch, hkv, n, d), -2, case["group"], levels)
        vq = K.kivi_quant_codes(src.values(torch.float16, batch, hkv, n, d), -1, case["group"], levels)
        st.update(q=src.values(torch.float16, batch, case["hq"], 1, d), kq=[t.contiguous() for t in kq], vq=[t.contiguous() for t in vq])
    elif kind == "vecstep":
        dtype = DTYPES[case["dtype"]]
        cfg = _vecinfer_config(src, case, case["key_bits"], case["key_sub"], fused_sdpa=True, fused_sdpa_memory_bound=True)
        cache = KVCacheFactory.create(cfg)
        _fill_context(cache, src, case, case["ctx"])
        st.update(cache=cache, tokens=_new_tokens(src, case, dtype))
    else:
        dtype, n = DTYPES[case["dtype"]], case["tokens"]
        config = _vecinfer_config(src, case, 12, 4) if case["method"] == "vecinfer" else KVCacheConfig(method=case["method"], head_dim=d)
        st.update(config=config, k=src.keys(dtype, batch, hkv, n, d), v=src.values(dtype, batch, hkv, n, d))
    return st


def _vecinfer_config(src, case, key_bits, key_sub, **more):
    """Codebooks at the scale of what they encode and smooth factors a kv head, as calibration gives them."""
    d, sample = case["d"], src.keys(torch.float32, 512, case["hkv"], case["d"])
    smooth = calibrate_smooth_factors(sample)
    tilde = apply_dual_transform_keys(sample.transpose(0, 1), smooth, walsh_hadamard_matrix(d, device="cuda"))
    return KVCacheConfig(method="vecinfer", head_dim=d, key_codebook_bits=key_bits, key_sub_dim=key_sub, smooth_factors=smooth,
                         key_codebook=src.normal(1 << key_bits, key_sub) * tilde.std(), value_codebook=src.normal(256, 8), **more)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("step", "vecstep"):
        cache, outs = st["cache"], []
        for t, (k, v, q) in enumerate(st["tokens"]):
            cache.update_and_fetch(k, v)
            if kind == "vecstep" or st["lengths"][t] is None:
                outs.append(cache.fused_sdpa(q, st["scale"]))
            else:
                outs.append(cache.fused_sdpa(q, st["scale"], lengths=st["lengths"][t]))
        cache.trim(STEPS)
        return outs
    if kind == "stack":
        cache, outs = st["cache"], []
        for k, v, q in st["tokens"]:
            for l, layer in enumerate(cache.layers):
                layer.update_and_fetch(k[l], v[l])
            outs.append(cache.fused_sdpa_all(q, st["scale"]))
        for layer in cache.layers:
            layer.trim(STEPS)
        return outs
    if kind == "prefill":
        cache = KVCacheFactory.create(st["config"])
        outs = []
        for k, v, q in st["chunks"]:
            cache.update_and_fetch(k, v)
            outs.append(cache.fused_sdpa(q, st["scale"], causal=True))
        return {"out": outs, "state": list(cache.state)}
    if kind == "flash":
        return K.flash_prefill_attend(st["q"], st["k"], st["v"], st["scale"])
    if kind == "scalar":
        return K.scalar_fused_decode_attend(st["q"], *st["kq"], *st["vq"], case["group"], st["scale"])
    return KVCacheFactory.create(st["config"]).update_and_fetch(st["k"], st["v"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _packed_bytes(case, tokens):
    """Codes, scale and zero of ``tokens`` packed tokens of one sequence of one layer, keys and values."""
    return 2 * case["hkv"] * tokens * case["d"] * (case["bits"] / 8 + 4 / case["group"])


def work(case):
    kind, d, b, hkv = case["kind"], case["d"], case["batch"], case["hkv"]
    if kind in ("step", "stack"):
        rows, ctx = STEPS * b * case.get("layers", 1), case["ctx"] + 1
        if case.get("ragged"):
            ctx = (ctx // 3 + ctx) // 2
        tail = min(ctx, RESIDUAL)
        return {"bytes": rows * (_packed_bytes(case, ctx - tail) + 2 * hkv * tail * d * 2 + 2 * hkv * d * 2 + 2 * case["hq"] * d * 2),
                "flops": rows * 4 * case["hq"] * d * ctx}
    n = case.get("tokens", case.get("ctx"))
    if kind == "prefill":
        return {"bytes": b * (2 * hkv * n * d * 2 + 2 * case["hq"] * n * d * 2 + _packed_bytes(case, n)),
                "flops": b * 4 * case["hq"] * d * n * (n + 1) / 2}
    if kind == "flash":
        return {"bytes": b * 2 * (hkv + case["hq"]) * n * d * 2, "flops": b * 4 * case["hq"] * d * n * (n + 1) / 2}
    if kind == "scalar":
        return {"bytes": b * (2 * hkv * n * d * (1 + 8 / case["group"]) + 2 * case["hq"] * d * 2), "flops": b * 4 * case["hq"] * d * n}
    if kind == "vecstep":
        index = (d // case["key_sub"]) * (4 if case["key_bits"] > 8 else 1) + d // 8
        return {"bytes": STEPS * b * (hkv * (n + 1) * index + 2 * hkv * d * 2 + 2 * case["hq"] * d * 2),
                "flops": STEPS * b * 4 * case["hq"] * d * (n + 1)}
    elements = b * hkv * n * d
    if case["method"] == "vecinfer":   # distances to every centroid as products of the sub-vectors
        return {"bytes": 2 * elements * 4, "flops": 2 * elements * (4096 + 256)}
    return {"bytes": 2 * elements * 4, "flops": 0}


def tolerance(case):
    """Four times the largest distance to the same path in float64 over the listed and forty drawn cases.  Seen, as 2-norm
    and as the largest single difference: decode in float16 2.4e-4 and 1.2e-3, in bfloat16 1.7e-3 and 3.9e-3 (the
    rounding of the output); causal calls over plain rows 2.6e-4 and 5.7e-3; prefill over the packed cache, whose rows
    are rounded to float16 once reconstructed, 8.9e-4 (bfloat16 1.85e-3) and 1.8e-2; VecInfer's reconstruction
    3.4e-4 and, where two centroids are equally near, 0.1; decode over VecInfer indices with the transform's sums in
    another order, which moves a few indices between equally near centroids, 2.6e-4 and 5.3e-3."""
    kind, half = case["kind"], case.get("dtype", "float16") == "float16"
    if kind == "fill":
        return {"rel": 1.4e-3 if half else 7e-3, "max": 0.4} if case["method"] == "vecinfer" else "exact"
    if kind == "prefill":
        return {"rel": 3.6e-3 if half else 7.4e-3, "max": 0.075}
    if kind == "flash":
        return {"rel": 1e-3, "max": 2.3e-2}
    most = 2.1e-2 if kind == "vecstep" else 5e-3 if half else 1.6e-2
    return {"rel": 1e-3 if half else 7e-3, "max": most}
