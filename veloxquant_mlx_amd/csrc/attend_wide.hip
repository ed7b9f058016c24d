// Attention of a few query rows over one long run of tokens whose channels a lane takes sixteen at a time: byte codes with
// float32 scale / zero (scalar_fused_decode_attend, veloxquant_mlx/metal/src/scalar_affine_attend.metal:57-174) and VecInfer
// codebook indices (VecInferKVCache.fused_sdpa, veloxquant_mlx/cache/vecinfer_cache.py:670-731).  Everything is computed in
// float32 on the vector unit; keys and values are rebuilt in registers.
//
// 32 / 8 heads of 128 channels, one query: byte codes of 2 x 8192 tokens 77 -> 21.2 us with the merge (42 MB, 2.0 TB/s);
// 4096 x 4 / 256 x 8 codebooks over 2 x 9001 tokens 203 us (copy of the indices, gather to float32, general kernel, merge) ->
// 22.5 us.  What bounds it is latency: a decode call reads a few tens of MB, so every wave has two or three units of tokens to do and
// waits for each.  Hence
//   * sixteen channels a lane: D / 16 lanes hold a token, a wave 64 / (D / 16) tokens at once, and the sums over a token's lanes
//     take two to four DPP adds a row (the general kernel in attend_rows.hip owns four channels a lane for byte codes: five);
//   * a wave takes a unit of 16 or 32 neighbouring tokens -- always inside one key group, so scale and zero are read once --
//     and asks for all codes of the unit before it uses the first;
//   * the running maximum moves once a unit;
//   * the centroids sit in LDS (64 KB for 4096 x 4, 8 KB for 256 x 8), and a token costs its indices: 144 bytes a token and
//     kv head at 128 channels instead of the 1024 + 1024 that a float32 copy takes to write and to read;
//   * the query transform of VecInfer, (q * smooth) @ Hadamard, is a fast transform of the block's rows in LDS.
// The slots' sums are added by halving exchanges (56 a wave for 4 x 16 sums over 8 slots; adding every sum over every slot
// takes 192).
// What is left is issue: with two waves a SIMD, 1300 instructions a unit and two or three units a wave, the instructions that run once
// count.  Row coordinates by comparison instead of division, exchanges by lane swaps instead of LDS permutes (80 waits in a
// row) and one pass over the block's partials took 3970 executed instructions a wave to 3520 (indices 3880 to 3435): byte codes of 2 x 8192 tokens
// 20.5 -> 18.7 us a launch, a call 22.9 -> 21.2, 2 x 9001 indices 20.9 -> 18.4 a launch (without the merge, 4 us).  Asking for the first unit ahead of tables and queries, eight pieces of the
// codebooks in flight, or a stretch of whole steps for every wave did not help (21.2, 21.9, 22.4 us): the waits are the other wave's turn.
#include <atomic>

#include "attend_rows.hpp"

namespace vq {

namespace {

constexpr int WD_THREADS = 512, WD_WAVES = WD_THREADS / 64;
constexpr float WD_LOG2E = 1.4426950408889634f, WD_LN2 = 0.6931471805599453f;
constexpr size_t WD_MAX_LDS = 144 * 1024;

struct WideArgs {
    const void *q;
    int q_dtype;
    int64_t Hq, Hkv, Sq, n, cap;     // n live tokens of cap
    float scale;
    int causal;
    int64_t window;
    const float *smooth;             // [smooth_rows, D] or null
    int smooth_rows;
    float hscale;                    // > 0: rows are multiplied by the Hadamard matrix of this magnitude
    int64_t split_len;
    int pq, tiles, group;            // group: query heads of a kv head
    float *ws;
};

// ---- byte codes, code * scale + zero; scales and zeros float32, value groups along the channels
struct ByteRows {
    const uint8_t *k, *v;
    const float *ks, *kz, *vs, *vz;
    int group;
    int64_t cap;

    struct Unit { float s[16], z[16]; };   // of the lane's channels in the unit's token group
    struct Raw { uint4 k, v; float vs, vz; };

    template <int D> __device__ void block_init(float *, int) const {}
    template <int D> __device__ __forceinline__ void unit(Unit &u, int64_t bh, int64_t t, int w) const {
        const int64_t gk = (cap + group - 1) / group, mi = (bh * gk + t / group) * D + w * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 a = *reinterpret_cast<const float4 *>(ks + mi + 4 * j), b = *reinterpret_cast<const float4 *>(kz + mi + 4 * j);
            u.s[4 * j] = a.x; u.s[4 * j + 1] = a.y; u.s[4 * j + 2] = a.z; u.s[4 * j + 3] = a.w;
            u.z[4 * j] = b.x; u.z[4 * j + 1] = b.y; u.z[4 * j + 2] = b.z; u.z[4 * j + 3] = b.w;
        }
    }
    template <int D> __device__ __forceinline__ void load(Raw &r, int64_t bh, int64_t t, int w) const {
        const int64_t row = bh * cap + t;
        r.k = *reinterpret_cast<const uint4 *>(k + row * D + w * 16);
        r.v = *reinterpret_cast<const uint4 *>(v + row * D + w * 16);
        const int gv = (D + group - 1) / group;
        const int64_t mi = row * gv + w * 16 / group;
        r.vs = vs[mi];
        r.vz = vz[mi];
    }
    static __device__ __forceinline__ void bytes(const uint4 &x, float (&o)[16]) {
        const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int j = 0; j < 16; ++j) o[j] = (float)((w[j / 4] >> (8 * (j % 4))) & 255u);
    }
    __device__ __forceinline__ void keys(const Raw &r, const Unit &u, const float *, float (&o)[16]) const {
        bytes(r.k, o);
#pragma unroll
        for (int j = 0; j < 16; ++j) o[j] = __builtin_fmaf(o[j], u.s[j], u.z[j]);
    }
    // values as codes: the caller multiplies the probability by the scale and sums the zeros apart
    static constexpr bool SCALED = true;
    __device__ __forceinline__ void values(const Raw &r, const float *, float (&o)[16]) const { bytes(r.v, o); }
    static __device__ __forceinline__ float vscale(const Raw &r) { return r.vs; }
    static __device__ __forceinline__ float vzero(const Raw &r) { return r.vz; }
};

// ---- codebook indices: sub-vectors of KSUB / VSUB channels, 8 or 32 bits an index
template <int KSUB, int VSUB> struct IndexRows {
    const void *k, *v;
    int k_u8, v_u8;
    const void *kcb, *vcb;
    int kcb_tag, vcb_tag, nk, nv;
    int64_t cap;

    static constexpr int NK = 16 / KSUB, NV = 16 / VSUB;   // indices of a lane
    struct Unit {};
    struct Raw { uint32_t k[NK], v[NV]; };

    // both codebooks as float32 into LDS, the keys' first
    template <int D> __device__ void block_init(float *lds, int tid) const {
        auto copy = [&](const void *src, int tag, int n, float *dst) {
            if (tag == VQ_F32 && ((uintptr_t)src & 15u) == 0) {
                for (int e = tid; e < n / 4; e += WD_THREADS) reinterpret_cast<float4 *>(dst)[e] = reinterpret_cast<const float4 *>(src)[e];
            } else {
                for (int e = tid; e < n; e += WD_THREADS) dst[e] = ar_ld(src, tag, e);
            }
        };
        copy(kcb, kcb_tag, nk * KSUB, lds);
        copy(vcb, vcb_tag, nv * VSUB, lds + nk * KSUB);
    }
    template <int D> __device__ __forceinline__ void unit(Unit &, int64_t, int64_t, int) const {}
    template <int N> static __device__ __forceinline__ void indices(const void *p, int u8, int64_t at, uint32_t (&o)[N]) {
        if (u8) {   // the same for the whole launch
            const uint8_t *b = (const uint8_t *)p + at;
            const uint32_t x = N == 4 ? *reinterpret_cast<const uint32_t *>(b) : *reinterpret_cast<const u16 *>(b);
#pragma unroll
            for (int j = 0; j < N; ++j) o[j] = (x >> (8 * j)) & 255u;
        } else {
            const uint32_t *b = (const uint32_t *)p + at;
            if constexpr (N == 4) {
                const uint4 x = *reinterpret_cast<const uint4 *>(b);
                o[0] = x.x; o[1] = x.y; o[2] = x.z; o[3] = x.w;
            } else {
                const uint2 x = *reinterpret_cast<const uint2 *>(b);
                o[0] = x.x; o[1] = x.y;
            }
        }
    }
    template <int D> __device__ __forceinline__ void load(Raw &r, int64_t bh, int64_t t, int w) const {
        const int64_t row = bh * cap + t;
        indices<NK>(k, k_u8, row * (D / KSUB) + w * NK, r.k);
        indices<NV>(v, v_u8, row * (D / VSUB) + w * NV, r.v);
    }
    // an index past the codebook takes its last entry, as the gather kernel does
    template <int SUB, int N> static __device__ __forceinline__ void gather(const uint32_t (&idx)[N], int n, const float *cb, float (&o)[16]) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t c = idx[i] < (uint32_t)n ? idx[i] : (uint32_t)n - 1u;
#pragma unroll
            for (int j = 0; j < SUB; j += 4) {
                const float4 x = *reinterpret_cast<const float4 *>(cb + c * SUB + j);
                o[i * SUB + j] = x.x; o[i * SUB + j + 1] = x.y; o[i * SUB + j + 2] = x.z; o[i * SUB + j + 3] = x.w;
            }
        }
    }
    __device__ __forceinline__ void keys(const Raw &r, const Unit &, const float *lds, float (&o)[16]) const { gather<KSUB, NK>(r.k, nk, lds, o); }
    static constexpr bool SCALED = false;
    __device__ __forceinline__ void values(const Raw &r, const float *lds, float (&o)[16]) const { gather<VSUB, NV>(r.v, nv, lds + nk * KSUB, o); }
    static __device__ __forceinline__ float vscale(const Raw &) { return 1.f; }
    static __device__ __forceinline__ float vzero(const Raw &) { return 0.f; }
};

// The wave's lanes OFF apart, without a trip through LDS: what both of them hold (in every lane, the lower one's first) ...
struct Both { float lo, hi; };
template <int OFF> __device__ __forceinline__ Both lanes_apart(float x) {
    if constexpr (OFF == 32 || OFF == 16) {
        const uint32_t u = __float_as_uint(x);
        const auto r = [&] {
            if constexpr (OFF == 32) return __builtin_amdgcn_permlane32_swap(u, u, false, false);
            else return __builtin_amdgcn_permlane16_swap(u, u, false, false);
        }();
        return {__uint_as_float(r[0]), __uint_as_float(r[1])};
    } else if constexpr (OFF == 8) {
        return {x, ar_dpp<0x128>(x)};   // row_ror 8
    } else {
        return {x, __shfl_xor(x, OFF)};
    }
}
// ... and a half-exchange: lanes with the bit OFF clear get the sum of both lanes' x, those with it set that of both lanes' y.
template <int OFF> __device__ __forceinline__ float exchange_add(float x, float y, bool upper) {
    if constexpr (OFF == 32 || OFF == 16) {
        const uint32_t u = __float_as_uint(x), v = __float_as_uint(y);
        const auto r = [&] {
            if constexpr (OFF == 32) return __builtin_amdgcn_permlane32_swap(u, v, false, false);
            else return __builtin_amdgcn_permlane16_swap(u, v, false, false);
        }();
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    } else {
        const float keep = upper ? y : x, give = upper ? x : y;
        return keep + (OFF == 8 ? ar_dpp<0x128>(give) : __shfl_xor(give, OFF));
    }
}
template <int OFF> __device__ __forceinline__ float slots_max(float x) {   // over the lanes OFF, 2 OFF, .. 32 apart
    const Both b = lanes_apart<OFF>(x);
    if constexpr (OFF == 32) return fmaxf(b.lo, b.hi);
    else return slots_max<2 * OFF>(fmaxf(b.lo, b.hi));
}
template <int OFF> __device__ __forceinline__ float slots_add(float x) {
    const Both b = lanes_apart<OFF>(x);
    if constexpr (OFF == 32) return b.lo + b.hi;
    else return slots_add<2 * OFF>(b.lo + b.hi);
}
// Sums a[0 .. T) over the 64 / LPT slots of a wave: at every exchange a lane keeps half of its sums and gives the other
// half away.  Returns the first of the T / (64 / LPT) sums that are left in a[0 ..].
template <int T, int OFF, int LPT> __device__ __forceinline__ int slots_reduce(float *a, int lane) {
    if constexpr (OFF < LPT) {
        return 0;
    } else {
        const bool upper = (lane & OFF) != 0;
#pragma unroll
        for (int j = 0; j < T / 2; ++j) a[j] = exchange_add<OFF>(a[j], a[j + T / 2], upper);
        return (upper ? T / 2 : 0) + slots_reduce<T / 2, OFF / 2, LPT>(a, lane);
    }
}

// The query rows of a block: `heads` heads of the group from h0 on, at consecutive positions from pos0 on.  At most AR_NR rows, so head
// and position of one take comparisons; as divisions, by every wave and for every row, they were a fifth of the instructions
// of a short run.
struct WideRows {
    int64_t base_row, Sq;   // row of (sequence, first head of the group, position 0); query positions
    int heads, h0, pos0, n;
    __device__ __forceinline__ int at(int r) const { return (r >= heads) + (r >= 2 * heads) + (r >= 3 * heads); }
    __device__ __forceinline__ bool valid(int r) const { return r < n && pos0 + at(r) < Sq; }
    __device__ __forceinline__ int64_t row(int r) const { return base_row + (int64_t)(h0 + r - at(r) * heads) * Sq + pos0 + at(r); }
};
static_assert(AR_NR <= 4, "WideRows::at");

template <int D, int NR, class Rows>
__global__ __launch_bounds__(WD_THREADS) void attend_wide_kernel(WideArgs a, Rows rows) {
    constexpr int LPT = D / 16, TPS = 64 / LPT;          // lanes of a token, tokens of a step
    constexpr int NS = TPS >= 16 ? 2 : 4, UNIT = TPS * NS;   // steps and tokens of a unit; 32 % UNIT == 0
    static_assert(32 % UNIT == 0, "a unit lies in one token group");
    extern __shared__ __align__(16) float s_dyn[];       // the rows' tables, after the loop the waves' partials
    __shared__ float s_q[NR][D];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sp = (int)blockIdx.x, nsplit = (int)gridDim.x;
    const uint32_t by = blockIdx.y, bh32 = by / (uint32_t)a.tiles, b = bh32 / (uint32_t)a.Hkv;   // (fewer than 65536 blocks)
    const int64_t bh = bh32, hkv = bh32 - b * (uint32_t)a.Hkv;
    const int w = lane % LPT, slot = lane / LPT;

    const int htiles = a.group > AR_NR ? (a.group + AR_NR - 1) / AR_NR : 1;
    const int t_in_bh = (int)(by - bh32 * (uint32_t)a.tiles);
    WideRows tile;
    tile.h0 = htiles > 1 ? (t_in_bh % htiles) * AR_NR : 0;
    tile.heads = htiles > 1 ? (a.group - tile.h0 < AR_NR ? a.group - tile.h0 : AR_NR) : a.group;
    tile.n = tile.heads * a.pq;
    tile.pos0 = (htiles > 1 ? t_in_bh / htiles : t_in_bh) * a.pq;
    tile.Sq = a.Sq;
    tile.base_row = ((int64_t)b * a.Hq + hkv * a.group) * a.Sq;

    rows.template block_init<D>(s_dyn, tid);
    for (int e = tid; e < NR * D; e += WD_THREADS) {
        const int r = e / D, d = e % D;
        float x = 0.f;
        if (tile.valid(r)) {
            x = ar_ld(a.q, a.q_dtype, tile.row(r) * D + d);
            if (a.smooth != nullptr) x *= a.smooth[(a.smooth_rows > 1 ? hkv * D : 0) + d];
        }
        s_q[r][d] = x;
    }
    __syncthreads();
    if (a.hscale > 0.f) {
        for (int h = 1; h < D; h <<= 1) {
            for (int e = tid; e < NR * D / 2; e += WD_THREADS) {
                const int r = e / (D / 2), i = e % (D / 2), lo = (i / h) * 2 * h + i % h;
                const float x = s_q[r][lo], y = s_q[r][lo + h];
                s_q[r][lo] = x + y;
                s_q[r][lo + h] = x - y;
            }
            __syncthreads();
        }
    }

    int64_t vis[NR], fst[NR], t_lo = INT64_MAX, t_hi = 0;   // row r sees tokens [fst, vis)
    float qs[NR][16], m[NR], l[NR], oz[NR], acc[NR * 16];
    const float mul = a.scale * WD_LOG2E * (a.hscale > 0.f ? a.hscale : 1.f);   // scores in log2 units
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        // queries align to the end of the tokens
        const int64_t upto = a.n - a.Sq + tile.pos0 + tile.at(r) + 1, from = upto - a.window;
        vis[r] = !tile.valid(r) ? 0 : a.causal ? upto : a.n;
        fst[r] = tile.valid(r) && a.window > 0 && from > 0 ? from : 0;
        if (tile.valid(r)) {
            t_lo = fst[r] < t_lo ? fst[r] : t_lo;
            t_hi = vis[r] > t_hi ? vis[r] : t_hi;
        }
        m[r] = -INFINITY;
        l[r] = oz[r] = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            qs[r][j] = s_q[r][w * 16 + j] * mul;
            acc[r * 16 + j] = 0.f;
        }
    }
    int64_t t0 = (int64_t)sp * a.split_len, t1 = t0 + a.split_len;
    if (t0 < t_lo) t0 = t_lo;
    if (t1 > t_hi) t1 = t_hi;
    bool masked = false;   // rows that see every token of [t0, t1) need no mask
#pragma unroll
    for (int r = 0; r < NR; ++r)
        if (tile.valid(r) && (fst[r] > t0 || vis[r] < t1)) masked = true;

    for (int64_t base = t0 / UNIT * UNIT + (int64_t)wave * UNIT; base < t1; base += WD_WAVES * UNIT) {
        typename Rows::Unit u;
        typename Rows::Raw raw[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int64_t t = base + i * TPS + slot;
            rows.template load<D>(raw[i], bh, t < a.n ? t : a.n - 1, w);
        }
        rows.template unit<D>(u, bh, base, w);
        const bool cut = masked || base < t0 || base + UNIT > t1;
        float s[NS][NR];
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            float k[16];
            rows.keys(raw[i], u, s_dyn, k);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                float x = 0.f, y = 0.f;
#pragma unroll
                for (int j = 0; j < 16; j += 2) {
                    x = __builtin_fmaf(qs[r][j], k[j], x);
                    y = __builtin_fmaf(qs[r][j + 1], k[j + 1], y);
                }
                s[i][r] = ar_slot_sum(x + y, LPT);
            }
            if (cut) {
                const int64_t t = base + i * TPS + slot;
#pragma unroll
                for (int r = 0; r < NR; ++r)
                    if (t < t0 || t >= t1 || t >= vis[r] || t < fst[r]) s[i][r] = -INFINITY;
            }
        }
        float mn[NR];
        bool up = false;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            mn[r] = m[r];
#pragma unroll
            for (int i = 0; i < NS; ++i) mn[r] = fmaxf(mn[r], s[i][r]);
            up |= mn[r] > m[r];
        }
        if (__any(up)) {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const float f = mn[r] == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[r] - mn[r]);   // 0 when m was -inf
                m[r] = mn[r];
                l[r] *= f;
                oz[r] *= f;
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[r * 16 + j] *= f;
            }
        }
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            float v[16];
            rows.values(raw[i], s_dyn, v);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const float p = s[i][r] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s[i][r] - m[r]);
                l[r] += p;
                float ps = p;
                if constexpr (Rows::SCALED) {
                    ps = p * Rows::vscale(raw[i]);
                    oz[r] = __builtin_fmaf(p, Rows::vzero(raw[i]), oz[r]);
                }
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[r * 16 + j] = __builtin_fmaf(v[j], ps, acc[r * 16 + j]);
            }
        }
    }

    // ---- the slots of the wave, then the waves of the block (a lane's probabilities are those of its token's other lanes)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const float mw = slots_max<LPT>(m[r]);
        const float f = m[r] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[r] - mw);
        l[r] = slots_add<LPT>(l[r] * f);
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[r * 16 + j] = Rows::SCALED ? (acc[r * 16 + j] + oz[r]) * f : acc[r * 16 + j] * f;
        m[r] = mw;
    }
    const int first = slots_reduce<NR * 16, 32, LPT>(acc, lane);
    __syncthreads();   // the tables are read no more
    float *part = s_dyn + wave * NR * (D + 2);
#pragma unroll
    for (int j = 0; j < NR * 16 / TPS; ++j) {
        const int e = first + j;
        part[(e / 16) * (D + 2) + 2 + w * 16 + e % 16] = acc[j];
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            part[r * (D + 2)] = m[r] * WD_LN2;   // -inf stays -inf
            part[r * (D + 2) + 1] = l[r];
        }
    }
    __syncthreads();
    for (int e = tid; e < NR * D; e += WD_THREADS) {   // a thread a sum; the first of a row also writes its maximum and weight
        const int r = e / D, c = e % D;
        if (!tile.valid(r)) continue;
        float mv[WD_WAVES], gm = -INFINITY, x = 0.f, den = 0.f;
#pragma unroll
        for (int v = 0; v < WD_WAVES; ++v) {
            mv[v] = s_dyn[(v * NR + r) * (D + 2)];
            gm = fmaxf(gm, mv[v]);
        }
#pragma unroll
        for (int v = 0; v < WD_WAVES; ++v) {
            const float *p = s_dyn + (v * NR + r) * (D + 2);
            const float f = mv[v] == -INFINITY ? 0.f : __expf(mv[v] - gm);
            if (mv[v] != -INFINITY) {
                x += p[2 + c] * f;
                den += p[1] * f;
            }
        }
        float *o = a.ws + (tile.row(r) * nsplit + sp) * (D + 2);
        o[2 + c] = x;
        if (c == 0) { o[0] = gm; o[1] = den; }
    }
}

// Splits: one block of eight waves a CU (the registers of four rows of sums leave room for one, the codebooks of the
// defaults in LDS for two), of at least 128 tokens.  A caller's own cut (`want`) is that of the vector kernel in attend_rows.hip, so
// that it means the same, and takes the same room for partials, whichever of the two runs.
void wide_splits(int64_t units, int64_t n, int want, int64_t &split_len, int &nsplit) {
    const int64_t least = want > 0 ? 256 : 128, gran = want > 0 ? 64 : 32;
    int64_t ns = want > 0 ? want : 256 / (units > 0 ? units : 1);
    const int64_t most = n > least ? n / least : 1;
    if (ns > most) ns = most;
    if (ns > 512) ns = 512;
    if (ns < 1) ns = 1;
    split_len = cdiv(cdiv(n, ns), gran) * gran;
    nsplit = (int)cdiv(n, split_len);
}

void wide_tiling(int64_t Hq, int64_t Hkv, int64_t Sq, int &pq, int &tiles) {
    AttendCall a = {};
    a.Hq = Hq;
    a.Hkv = Hkv;
    a.Sq = Sq;
    rows_tiling(a, pq, tiles);
}

template <int D, int NR, class Rows>
void launch_wide_rows(const WideArgs &w, const Rows &rows, dim3 grid, size_t tables, hipStream_t st) {
    const size_t parts = (size_t)WD_WAVES * NR * (D + 2) * sizeof(float), lds = tables > parts ? tables : parts;
    if (lds > 48 * 1024) {   // more dynamic LDS than the default limit has to be allowed once per kernel and device
        static std::atomic<bool> allowed[64] = {};   // a second thread that gets here first repeats the same call
        int dev = 0;
        (void)hipGetDevice(&dev);
        if (dev < 0 || dev >= 64 || !allowed[dev].load(std::memory_order_acquire)) {
            (void)hipFuncSetAttribute((const void *)attend_wide_kernel<D, NR, Rows>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)WD_MAX_LDS);
            if (dev >= 0 && dev < 64) allowed[dev].store(true, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL((attend_wide_kernel<D, NR, Rows>), grid, dim3(WD_THREADS), lds, st, w, rows);
}

template <int D, class Rows> void launch_wide_d(const WideArgs &w, const Rows &rows, dim3 grid, size_t tables, hipStream_t st) {
    const int64_t R = w.Hq / w.Hkv;
    switch ((int)((R > AR_NR ? AR_NR : R) * w.pq)) {   // rows of the largest tile
        case 1: launch_wide_rows<D, 1>(w, rows, grid, tables, st); break;
        case 2: launch_wide_rows<D, 2>(w, rows, grid, tables, st); break;
        case 3: launch_wide_rows<D, 3>(w, rows, grid, tables, st); break;
        default: launch_wide_rows<D, 4>(w, rows, grid, tables, st); break;
    }
}

template <class Rows> void launch_wide(const WideArgs &w, const Rows &rows, int64_t B, int64_t D, int nsplit, size_t tables, hipStream_t st) {
    const dim3 grid((unsigned)nsplit, (unsigned)(B * w.Hkv * w.tiles));
    if (D == 64) launch_wide_d<64>(w, rows, grid, tables, st);
    else if (D == 128) launch_wide_d<128>(w, rows, grid, tables, st);
    else launch_wide_d<256>(w, rows, grid, tables, st);
}

bool wide_head(int64_t D) { return D == 64 || D == 128 || D == 256; }
// Query rows of a kv head.  Every tile of four reads the tokens again, which for byte codes ends at the few rows of a draft
// to be verified; for indices anything below a prefill-sized call (256 rows) is cheaper than a float32 copy of the context
// (32 / 8 heads of 128 channels, 4 x 16384 tokens, 16 rows: 142 us, 1287 us through the copy).
constexpr int64_t WD_MAX_ROWS = 16, WD_MAX_INDEX_ROWS = 255;

}  // namespace

// Byte codes as a whole context: no tail, no protected rows, one length.  Every lane's sixteen channels lie in one value
// group and every unit of tokens in one key group, and all pieces are 16-byte aligned.  The batch counts only where the grid ends
// (grid y, as in rows_kernel_supported): layers stacked into one call take the kernel that a call a layer takes (600 sequences
// of 32 / 8 heads of 128 channels, 4096 tokens: 5970 us in attend_rows.hip, 1403 here; 4607 x 8 / 8 of 64, 512 tokens 1602 and 614).
bool wide_kernel_supported(const AttendCall &a) {
    if (a.Hkv < 1 || a.Hq % a.Hkv != 0 || (a.Hq / a.Hkv) * a.Sq > WD_MAX_ROWS) return false;
    int pq, tiles;
    rows_tiling(a, pq, tiles);
    // Many tiles over a few tokens each: a block of eight waves has work for one or two of them, and the four-wave blocks of
    // attend_rows.hip are done sooner.  us there / here, 128 channels, 1024 tiles: 16 tokens 33 / 41, 33 38 / 41, 48 45 / 42;
    // 3200: 33 tokens 93 / 126, 64 115 / 122, 80 143 / 130; 512: 16 tokens 21 / 23, 33 23 / 23; 256: 16 tokens 18 / 14.  64 channels
    // reach it at twice the tokens (1024 tiles: 64 tokens 33 / 34, 80 41 / 35; 3200: 64 tokens 77 / 100, 160 130 / 120), 256 at half
    // (1600: 16 tokens 45 / 60, 33 67 / 67).
    // A caller's own cut keeps its kernel whatever the batch.
    const int64_t blocks = a.B * a.Hkv * (int64_t)tiles;
    if (a.num_splits == 0 && blocks > 256 && a.n_packed * a.D <= (blocks > 1536 ? 8192 : 4608)) return false;
    return a.num_splits >= 0 && a.n_packed > 0 && a.n_tail == 0 && a.pack_bits == 8 && a.v_layout == VQ_V_CHANNEL_PACKED &&
           a.meta_dtype == VQ_F32 && wide_head(a.D) && a.group % 32 == 0 && a.packed_lens == nullptr && a.k_new == nullptr &&
           a.sink_k == nullptr && a.scale > 0.f && blocks <= 65535 &&
           (((uintptr_t)a.k_packed | (uintptr_t)a.v_packed | (uintptr_t)a.k_scale | (uintptr_t)a.k_zero) & 15u) == 0;
}

void plan_attend_wide(const AttendCall &a, AttendPlan &p) {
    rows_tiling(a, p.pq, p.tiles);
    wide_splits(a.B * a.Hkv * p.tiles, a.n_packed, a.num_splits, p.split_len, p.nsplit);
    p.nparts = p.nsplit;
}

void launch_attend_wide(const AttendCall &a, const AttendPlan &p) {
    const WideArgs w = {a.q, a.q_dtype, a.Hq, a.Hkv, a.Sq, a.n_packed, a.cap_tokens, a.scale, a.causal, a.sliding_window,
                        nullptr, 1, 0.f, p.split_len, p.pq, p.tiles, (int)(a.Hq / a.Hkv), (float *)a.workspace};
    const ByteRows rows = {(const uint8_t *)a.k_packed, (const uint8_t *)a.v_packed, (const float *)a.k_scale, (const float *)a.k_zero,
                           (const float *)a.v_scale, (const float *)a.v_zero, a.group, a.cap_tokens};
    launch_wide(w, rows, a.B, a.D, p.nsplit, 0, (hipStream_t)a.stream);
}

// ---------------------------------------------------------------------------
// VecInfer indices
// ---------------------------------------------------------------------------
namespace {

size_t index_tables(const vq_index_attend_args &a) {
    return ((size_t)a.n_k_centroids * a.k_sub_dim + (size_t)a.n_v_centroids * a.v_sub_dim) * sizeof(float);
}

int validate_index(const vq_index_attend_args *a, const char *fn) {
    VQ_REQUIRE(a != nullptr, VQ_ERR_INVALID, "%s: null argument block", fn);
    VQ_REQUIRE(a->B >= 1 && a->Hq >= 1 && a->Hkv >= 1 && a->Sq >= 1 && a->D >= 1, VQ_ERR_INVALID, "%s: q must be 4D with positive sizes", fn);
    VQ_REQUIRE(a->Hq % a->Hkv == 0, VQ_ERR_INVALID, "%s: H_q=%lld must be a multiple of H_kv=%lld", fn, (long long)a->Hq, (long long)a->Hkv);
    VQ_REQUIRE(a->n_tokens >= 1 && a->cap_tokens >= a->n_tokens, VQ_ERR_INVALID, "%s: need 1 <= n_tokens <= cap_tokens", fn);
    VQ_REQUIRE(!a->causal || a->Sq <= a->n_tokens, VQ_ERR_INVALID, "%s: S_q=%lld exceeds S_kv=%lld; queries align to the tail of the KV cache",
               fn, (long long)a->Sq, (long long)a->n_tokens);
    VQ_REQUIRE(a->sliding_window >= 0, VQ_ERR_INVALID, "%s: negative sliding window", fn);
    VQ_REQUIRE(is_float_tag(a->q_dtype) && is_float_tag(a->out_dtype) && is_float_tag(a->k_cb_dtype) && is_float_tag(a->v_cb_dtype),
               VQ_ERR_INVALID, "%s: unsupported float dtype", fn);
    VQ_REQUIRE((a->k_idx_dtype == VQ_U8 || a->k_idx_dtype == VQ_I32) && (a->v_idx_dtype == VQ_U8 || a->v_idx_dtype == VQ_I32),
               VQ_ERR_INVALID, "%s: indices must be uint8 or int32", fn);
    VQ_REQUIRE(a->n_k_centroids >= 1 && a->n_v_centroids >= 1, VQ_ERR_INVALID, "%s: empty codebook", fn);
    VQ_REQUIRE(a->smooth == nullptr || a->smooth_rows == 1 || a->smooth_rows == a->Hkv, VQ_ERR_INVALID, "%s: smooth must have 1 or H_kv rows", fn);
    VQ_REQUIRE(wide_head(a->D) && (a->k_sub_dim == 4 || a->k_sub_dim == 8) && a->v_sub_dim == 8 && a->scale > 0.f &&
                   a->n_k_centroids <= 65536 && a->n_v_centroids <= 65536 && index_tables(*a) <= WD_MAX_LDS &&
                   (a->Hq / a->Hkv) * a->Sq <= WD_MAX_INDEX_ROWS,
               VQ_ERR_UNSUPPORTED, "%s: shapes outside what the kernel covers", fn);
    // the batch counts only where the grid ends (32 / 8 heads of 128 channels, one row, 4096 x 4 codebooks: 40 x 9001 tokens 331 us,
    // 3426 through a copy of the context; 40 x 300 34 and 158)
    int pq, tiles;
    wide_tiling(a->Hq, a->Hkv, a->Sq, pq, tiles);
    VQ_REQUIRE(a->B * a->Hkv * (int64_t)tiles <= 65535, VQ_ERR_UNSUPPORTED, "%s: too many (sequence, kv head, row tile) blocks", fn);
    return VQ_OK;
}

void plan_index(const vq_index_attend_args &a, int &pq, int &tiles, int64_t &split_len, int &nsplit) {
    wide_tiling(a.Hq, a.Hkv, a.Sq, pq, tiles);
    wide_splits(a.B * a.Hkv * tiles, a.n_tokens, 0, split_len, nsplit);
}

}  // namespace

}  // namespace vq

using namespace vq;

extern "C" size_t vq_vecinfer_attend_indices_workspace(const vq_index_attend_args *a) {
    if (validate_index(a, "vq_vecinfer_attend_indices_workspace") != VQ_OK) return 0;
    int pq, tiles, nsplit;
    int64_t len;
    plan_index(*a, pq, tiles, len, nsplit);
    return (size_t)(a->B * a->Hq * a->Sq) * (size_t)nsplit * (size_t)(a->D + 2) * sizeof(float);
}

extern "C" int vq_vecinfer_attend_indices(const vq_index_attend_args *a) {
    const char *fn = "vq_vecinfer_attend_indices";
    const int rc = validate_index(a, fn);
    if (rc != VQ_OK) return rc;
    VQ_REQUIRE(a->q && a->out && a->k_idx && a->v_idx && a->k_codebook && a->v_codebook, VQ_ERR_INVALID, "%s: null pointer", fn);
    VQ_REQUIRE((((uintptr_t)a->k_idx | (uintptr_t)a->v_idx) & 15u) == 0, VQ_ERR_UNSUPPORTED, "%s: index buffers must be 16-byte aligned", fn);
    int pq, tiles, nsplit;
    int64_t len;
    plan_index(*a, pq, tiles, len, nsplit);
    const int64_t rows = a->B * a->Hq * a->Sq;
    const size_t need = (size_t)rows * (size_t)nsplit * (size_t)(a->D + 2) * sizeof(float);
    VQ_REQUIRE(a->workspace && a->workspace_bytes >= need, VQ_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", fn, need,
               a->workspace_bytes);
    hipStream_t st = (hipStream_t)a->stream;
    const WideArgs w = {a->q, a->q_dtype, a->Hq, a->Hkv, a->Sq, a->n_tokens, a->cap_tokens, a->scale, a->causal, a->sliding_window,
                        a->smooth, a->smooth_rows, a->hadamard_scale, len, pq, tiles, (int)(a->Hq / a->Hkv), (float *)a->workspace};
    auto run = [&](auto r) {
        r.k = a->k_idx; r.v = a->v_idx;
        r.k_u8 = a->k_idx_dtype == VQ_U8; r.v_u8 = a->v_idx_dtype == VQ_U8;
        r.kcb = a->k_codebook; r.vcb = a->v_codebook;
        r.kcb_tag = a->k_cb_dtype; r.vcb_tag = a->v_cb_dtype;
        r.nk = a->n_k_centroids; r.nv = a->n_v_centroids;
        r.cap = a->cap_tokens;
        launch_wide(w, r, a->B, a->D, nsplit, index_tables(*a), st);
    };
    if (a->k_sub_dim == 4) run(IndexRows<4, 8>{});
    else run(IndexRows<8, 8>{});
    VQ_HIP_CHECK_LAUNCH(fn);
    launch_merge_splits((const float *)a->workspace, rows, nsplit, a->D, a->out, a->out_dtype, st);
    VQ_HIP_CHECK_LAUNCH(fn);
    return VQ_OK;
}
