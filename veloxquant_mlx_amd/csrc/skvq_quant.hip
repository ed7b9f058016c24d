// SKVQ clipped group quantisation round trip for gfx950.
//
// Per token row and per group of `group` consecutive (optionally permuted) channels
// (veloxquant_mlx/quantizers/skvq.py:105-183, float32, one rounding per operation):
//   mid = (gmax + gmin) * 0.5,  rng = gmax - gmin
//   for every clip factor a:  lo = mid - (a * rng) * 0.5,  scale = max((a * rng) / levels, 1e-8)
//                             code = clamp(rint((x - lo) / scale), 0, levels),  xhat = code * scale + lo
//                             err  = sum((xhat - x)^2) / group        (summed left to right)
//   the first a with the smallest err wins; out = cast(xhat of that a).
// A ragged last group is padded with the row's last (permuted) channel, as the reference pads.
// With a permutation, group j of a row of head h holds channels perm[h][j*group .. ], and the
// result goes back to the channels it came from (the inverse gather of
// veloxquant_mlx/cache/skvq_cache.py:236-251).
//
// One thread owns one group.  A block first stages its rows in LDS as float32 (stride group + 1
// words between groups, so the threads of a wave walk different banks), then every thread scans
// its group once per clip factor (held in registers for groups of 32 and 64, out of LDS otherwise),
// overwrites it with the winning reconstruction, and the block writes the rows back.  Staging completes before the first store, so out may alias x.
#include "common.hpp"

namespace vq {

constexpr int SK_THREADS = 256;
constexpr int SK_MAX_ALPHAS = 8;
constexpr int SK_AHEAD = 4;    // rows a thread requests at a time

struct SkAlphas { float a[SK_MAX_ALPHAS]; int n; };
// what differs between the tensors of a launch (blockIdx.z); perm / inv as void: the order kernel writes them
struct SkSide { const void *x; void *out; int32_t *perm, *inv; float levels; };
struct SkSides { SkSide t[2]; };

// clamp(rint((x - lo) / sc), 0, levels) without an IEEE division on the common path.  t = x - lo is
// rounded once, as in the reference; q0 = t * rcp(sc) lies within 2.5 ulp (1.5e-7 relative) of the
// correctly rounded quotient, so rint(q0) is the reference's code unless q0 sits that close to a tie
// k + 0.5 -- a lane within 1e-6 * (|q0| + 1) of one takes the true division instead.
__device__ __forceinline__ float sk_code(float x, float lo, float sc, float rs, float levels) {
    const float t = __fsub_rn(x, lo);
    const float q0 = __fmul_rn(t, rs);
    float r = rintf(q0);
    if (fabsf(q0 - r) >= 0.5f - 1e-6f * (fabsf(q0) + 1.0f)) r = rintf(__fdiv_rn(t, sc));
    return fminf(fmaxf(r, 0.f), levels);
}

// Eight codes at a time with one tie limit for the whole call and one branch: when any lane of the wave
// has any of its eight q0 within `tie` of a half, all eight are formed again by true division (rare, and
// the same value wherever q0 was not close).  Outside |q0| <= levels + 1 the clamp decides whatever the
// rounding does; inside it q0 is within 1.5e-7 * (levels + 1) of the true quotient, less than the
// 1e-6 * (levels + 2) by which `tie` stays below one half.
__device__ __forceinline__ void sk_codes8(const float *x, float (&q)[8], float lo, float sc, float rs, float levels, float tie) {
    float far = 0.f, dist[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float q0 = __fmul_rn(__fsub_rn(x[j], lo), rs);
        q[j] = rintf(q0);
        dist[j] = fabsf(q0 - q[j]);
        far = fmaxf(far, dist[j]);
    }
    if (__builtin_amdgcn_ballot_w64(far >= tie) != 0) {   // exact ties are common with 16-bit inputs: only the codes some lane is unsure of
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (__builtin_amdgcn_ballot_w64(dist[j] >= tie) != 0) q[j] = rintf(__fdiv_rn(__fsub_rn(x[j], lo), sc));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = __builtin_amdgcn_fmed3f(q[j], 0.f, levels);   // a NaN becomes 0, as with fmaxf / fminf
}

// eight consecutive elements as one (16-bit types) or two (float32) 16-byte accesses
template <typename T> struct Vec8 {
    struct Raw { uint4 w[sizeof(T) / 2]; };   // as loaded
    static __device__ __forceinline__ Raw request(const T *p) {
        Raw r;
#pragma unroll
        for (int i = 0; i < (int)sizeof(T) / 2; ++i) r.w[i] = reinterpret_cast<const uint4 *>(p)[i];
        return r;
    }
    static __device__ __forceinline__ void unpack(const Raw &r, float (&v)[8]) {
        const T *e = reinterpret_cast<const T *>(&r);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = Elem<T>::ld(e + k);
    }
    static __device__ __forceinline__ void ld(const T *p, float (&v)[8]) {
        if constexpr (sizeof(T) == 4) {
            const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
            union { uint4 u; T e[8]; } w;
            w.u = *reinterpret_cast<const uint4 *>(p);
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = Elem<T>::ld(&w.e[k]);
        }
    }
    static __device__ __forceinline__ void st(T *p, const float (&v)[8]) {
        if constexpr (sizeof(T) == 4) {
            *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<float4 *>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
        } else {
            union { uint4 u; T e[8]; } w;
#pragma unroll
            for (int k = 0; k < 8; ++k) Elem<T>::st(&w.e[k], v[k]);
            *reinterpret_cast<uint4 *>(p) = w.u;
        }
    }
};

// The clip factors whose error can be the smallest, as bits.  The stated error of a factor -- codes by division, every step
// rounded, squares added left to right -- costs ten operations a value and a division where a code is near a tie; five give r = sc * sqrt(sum((t - q)^2)) with
// t = (x - lo) / sc in one fma and q = clamp(rint(t)), which is close enough to rule out
// all factors but one in 99.6 % of the groups at 4 bits (a 4100-token prompt of 8 x 8 heads, both tensors with their orders: 243 ->
// 230 us, 206 now; what is left is vector issue, 93 % of the SIMD-busy cycles).
// How close (u = 2^-24, W = levels * sc, M the largest |x|, so |lo| <= M and |x - lo| <= rng to within a few u * M):
//   * the stated difference d = q * sc + lo - x of a code has an error of u (3 W + 3 M);
//   * t has an error of u (2 rng + M) / sc (1 / sc is good to u after the Newton step), the stated quotient one of 2 u rng / sc;
//   * the stated code is the nearest of 0 .. levels to its quotient, q the nearest to t, and the distance to the nearest of a set of
//     numbers changes by no more than the number does: sc |t - q| and the stated |d| differ by u (4 rng + M) for the two errors above;
//   * t - q is rounded where the clamp moved q: u rng.
// So every |d| is within u (3 W + 4 M + 5 rng) of sc |t - q|.  The factor 1 clips nothing, and its q stays unclamped.  That is another number only where t
// lies half a code outside [0, levels] or further, and then both distances are at most that of t to the end.  How far out: mid, the range, lo and the
// scale are rounded, u M, u rng, u (M + rng / 2) and u W, so x - lo lies within u (2 M + 1.5 rng + W) of [0, W] (a scale raised to 1e-8: W is longer than
// the range, and only 0 is passed), and t by its own error, u (2 rng + M), further -- over many codes where the range is a few last places of
// M.  With it the distance is u (4 W + 7 M + 8 rng) at most.
// By the triangle inequality the roots of the two sums differ by at most sqrt(GROUP) times these; the sums' own rounding and the root cost (GROUP + 6) u
// relative.  The bounds below are these with a seventh of M and 6 u rng to spare (over groups of magnitudes 1e-3 to 1e5 and ranges down to 1e-9 of
// them the roots differ by a quarter of the bound at most).  Errors below 1e-15, where squares lose bits, stay open, and so does everything at magnitudes
// whose squares could overflow and for values that are not numbers.  `low` is the group's own memory, read before.
// best_lo / best_sc: of the one factor that is open, if it is one.
template <int GROUP, class Factor>
__device__ __forceinline__ uint32_t sk_open_factors(const float *xv, float *low, const SkAlphas &al, const Factor &factor, float M, float rng,
                                                    float levels, float &best_lo, float &best_sc) {
    constexpr float U = 5.9604645e-8f, REL = (GROUP + 16) * U, ROOT = GROUP <= 32 ? 5.66f : 8.01f;
    static_assert(GROUP >= SK_MAX_ALPHAS && GROUP <= 64, "a group has a word for every factor");
    float high = INFINITY;   // the smallest upper bound of a factor's error
    for (int k = 0; k < al.n; ++k) {
        float lo, sc, s0 = 0.f;
        factor(k, lo, sc);
        float rs = __builtin_amdgcn_rcpf(sc);
        rs = __builtin_fmaf(__builtin_fmaf(-sc, rs, 1.f), rs, rs);
        const float c = -lo * rs;
        if (al.a[k] == 1.f) {   // nothing is clipped, see above (207.2 -> 205.9 us)
#pragma unroll
            for (int j = 0; j < GROUP; ++j) {
                const float t = __builtin_fmaf(xv[j], rs, c);
                const float d = t - __builtin_rintf(t);
                s0 = __builtin_fmaf(d, d, s0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < GROUP; ++j) {
                const float t = __builtin_fmaf(xv[j], rs, c);
                const float d = t - __builtin_amdgcn_fmed3f(__builtin_rintf(t), 0.f, levels);
                s0 = __builtin_fmaf(d, d, s0);
            }
        }
        const float r = sc * __builtin_amdgcn_sqrtf(s0);
        const float off = ROOT * U * (4.f * levels * sc + 8.f * M + 14.f * rng) + 1e-15f;
        low[k] = s0 < 1e30f ? r * (1.f - REL) - off : -INFINITY;   // (a factor near 0 can overflow the sum)
        const float up = r * (1.f + REL) + off;
        if (up < high) { high = up; best_lo = lo; best_sc = sc; }   // (this factor stays open)
    }
    if (!(M < 1e15f)) high = INFINITY;
    uint32_t open = 0;
    for (int k = 0; k < al.n; ++k) open |= (low[k] > high ? 0u : 1u) << k;
    return open;
}

// ERR: the squared error of the float32 reconstruction instead of the reconstruction, the stored channel order
// (blockIdx.y 0) against the order `perm` (1), of the tensor blockIdx.z: err[((2 z + y) n_rows + row) tpr + piece] takes the double-precision sum over
// the channels of one thread's pieces, in stored channel order for both.
template <typename T, int GROUP, bool ERR>   // GROUP > 0: the group size, known at compile time; 0: any
__global__ __launch_bounds__(SK_THREADS)
void skvq_roundtrip_kernel(SkSides sides, double *__restrict__ err, int64_t n_bh, int64_t H, int64_t r, int64_t D,
                           int64_t x_stride_bh, int64_t out_stride_bh,
                           int group, uint64_t group_magic, int G, int rows_pb, int tpr, bool vec, SkAlphas al) {
    extern __shared__ float s_x[];
    const SkSide side = sides.t[ERR ? blockIdx.z : 0];
    const T *x = (const T *)side.x;
    T *out = (T *)side.out;
    const int32_t *__restrict__ perm = side.perm, *__restrict__ inv = side.inv;
    const float levels = side.levels;
    if (ERR && blockIdx.y == 0) perm = inv = nullptr;
    const int tid = threadIdx.x;
    const int gstride = group + 1, Dp = G * group;
    const int64_t row0 = (int64_t)blockIdx.x * rows_pb, n_rows = n_bh * r;   // n_rows < 2^31 (checked by the caller)

    // A thread moves pieces of eight consecutive channels: tpr threads side by side cover a row, the
    // block covers rpp rows per pass.  Rows that can move as 16-byte pieces (`vec`) do so; under a
    // channel order this needs the inverse order (channel -> place), which turns the gather into a
    // scatter inside LDS.  Without it, or with an odd head_dim, a piece is eight single-channel accesses
    // (gathers within the row's cache lines).
    // (Passing permuted rows through a second LDS image, to keep global accesses vectorised, measured
    // slower than these gathers: 0.92 ms against 0.79 ms on 16 x 8 x 8192 rows of 128 channels.)
    //
    // Where a row is one piece per thread (tpr * 8 >= Dp) a thread meets the same eight channels in every
    // row, so their LDS words -- a division by the group size and, under an order, a table look-up each --
    // are worked out once per head, not once per element; (sequence, head) and token of a row follow from
    // those of the block's first row by counting, not by dividing.
    const int lr_base = tid / tpr, cq = tid - lr_base * tpr, rpp = (int)blockDim.x / tpr;
    auto pos = [&](int j) {                        // LDS word of (permuted) channel j within a row
        if constexpr (GROUP > 0) return j + j / GROUP;
        const int gi = (int)(((uint64_t)(uint32_t)j * group_magic) >> 32);   // j / group
        return gi * gstride + (j - gi * group);
    };
    const bool scatter = vec && inv, one_piece = tpr * 8 >= Dp;
    const uint32_t bh_first = (uint32_t)row0 / (uint32_t)r, t_first = (uint32_t)row0 - bh_first * (uint32_t)r;
    const uint32_t head_first = bh_first % (uint32_t)H;
    struct Where { uint32_t bh, t, head; };
    auto where = [&](int lr) {                     // rows_pb rows span few (sequence, head) pairs
        Where w{bh_first, t_first + (uint32_t)lr, head_first};
        while (w.t >= (uint32_t)r) { w.t -= (uint32_t)r; ++w.bh; w.head = w.head + 1 == (uint32_t)H ? 0u : w.head + 1; }
        return w;
    };
    int off[8], fill_k = -1;
    uint32_t off_head = ~0u;
    auto place = [&](uint32_t head, int c0) {      // LDS words of channels (or places) c0 .. c0 + 7 of a row of `head`
        if (one_piece && head == off_head) return;
        off_head = head;
        fill_k = -1;
        const int32_t *iv = scatter ? inv + (int64_t)head * D : nullptr;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int c = c0 + k, j = (iv && c < (int)D) ? iv[c] : c;
            off[k] = pos(j);
            if (iv && j == (int)D - 1 && Dp > (int)D) fill_k = k;   // the order's last channel also fills a ragged last group
        }
    };
    // Rows of one piece a thread and whole groups of 32 or 64: SK_AHEAD of them are requested before the first is put in its
    // place (8 x 8 heads of 4091 rows, in place, five factors and orders: 80 us, 83 us with one request at a time; stored order
    // 69 and 74 us).  Elsewhere it costs: a ragged last group leaves its pad to threads that then wait for a second loop
    // (80 channels, groups of 32, 1024 rows 13.7 -> 16.1 us), and the kernel for any group is no quicker for it (64 x 1024 rows
    // of 256 channels, groups of 16 32.2 -> 35.5).
    const bool ahead = GROUP > 0 && vec && one_piece && Dp == (int)D;
    if (ahead) {
        const int c0 = cq * 8;
        for (int lr0 = lr_base; lr0 < rows_pb && lr_base < rpp; lr0 += SK_AHEAD * rpp) {
            typename Vec8<T>::Raw raw[SK_AHEAD];
            uint32_t head[SK_AHEAD];
#pragma unroll
            for (int i = 0; i < SK_AHEAD; ++i) {
                const int lr = lr0 + i * rpp;
                if (lr >= rows_pb || row0 + lr >= n_rows) continue;
                const Where w = where(lr);
                head[i] = w.head;
                raw[i] = Vec8<T>::request(x + (int64_t)w.bh * x_stride_bh + (int64_t)w.t * D + c0);
            }
#pragma unroll
            for (int i = 0; i < SK_AHEAD; ++i) {
                const int lr = lr0 + i * rpp;
                if (lr >= rows_pb || row0 + lr >= n_rows) continue;
                float v[8];
                Vec8<T>::unpack(raw[i], v);
                place(head[i], c0);
                float *dst = s_x + lr * G * gstride;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    dst[off[k]] = v[k];
                    if (k == fill_k)
                        for (int jp = (int)D; jp < Dp; ++jp) dst[pos(jp)] = v[k];
                }
            }
        }
    }
    for (int lr = lr_base; !ahead && lr < rows_pb && lr_base < rpp; lr += rpp) {
        if (row0 + lr >= n_rows) continue;
        const Where w = where(lr);
        const T *src = x + (int64_t)w.bh * x_stride_bh + (int64_t)w.t * D;
        const int32_t *pm = perm ? perm + (int64_t)w.head * D : nullptr;
        float *dst = s_x + lr * G * gstride;
        for (int c0 = cq * 8; c0 < Dp; c0 += tpr * 8) {
            float v[8];
            place(w.head, c0);
            if (scatter) {      // stored-order piece, every channel dropped at its place in the head's order
                if (c0 < D) {
                    Vec8<T>::ld(src + c0, v);
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        dst[off[k]] = v[k];
                        if (k == fill_k)
                            for (int jp = (int)D; jp < Dp; ++jp) dst[pos(jp)] = v[k];
                    }
                }
                continue;
            }
            if (vec && c0 < D) {
                Vec8<T>::ld(src + c0, v);
            } else {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int j = c0 + k, c = j < D ? j : (int)D - 1;
                    v[k] = Elem<T>::ld(src + (pm ? pm[c] : c));
                }
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (c0 + k < Dp) dst[off[k]] = v[k];
        }
    }
    __syncthreads();

    if (tid < rows_pb * G && row0 + tid / G < n_rows) {
        float *p = s_x + tid * gstride;
        if constexpr (GROUP > 0) {
            // the group in registers: LDS is read once and written once, and the clip search runs
            // as straight-line code over GROUP values per factor
            float xv[GROUP];
#pragma unroll
            for (int j = 0; j < GROUP; ++j) xv[j] = p[j];
            float mn = xv[0], mx = xv[0];
#pragma unroll
            for (int j = 1; j < GROUP; ++j) { mn = fminf(mn, xv[j]); mx = fmaxf(mx, xv[j]); }
            const float mid = __fmul_rn(__fadd_rn(mx, mn), 0.5f), rng = __fsub_rn(mx, mn);
            const float tie = 0.5f - 1e-6f * (levels + 2.0f);
            auto factor = [&](int k, float &lo, float &sc) {
                const float ar = __fmul_rn(al.a[k], rng);
                lo = __fsub_rn(mid, __fmul_rn(ar, 0.5f));
                sc = fmaxf(__fdiv_rn(ar, levels), 1e-8f);
            };
            float best_err = 0.f, best_lo = 0.f, best_sc = 1.f;
            uint32_t open = 1u;   // the factors that can be the winner
            if (al.n > 1) open = sk_open_factors<GROUP>(xv, p, al, factor, fmaxf(fabsf(mn), fabsf(mx)), rng, levels, best_lo, best_sc);
            else factor(0, best_lo, best_sc);
            const bool several = (open & (open - 1)) != 0;
            bool first = true;
            for (int k = 0; k < al.n; ++k) {
                const bool mine = several && ((open >> k) & 1u);
                if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
                float lo, sc, sum = 0.f;
                factor(k, lo, sc);
                const float rs = __builtin_amdgcn_rcpf(sc);
#pragma unroll
                for (int j0 = 0; j0 < GROUP; j0 += 8) {
                    float q[8];
                    sk_codes8(xv + j0, q, lo, sc, rs, levels, tie);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float d = __fsub_rn(__fadd_rn(__fmul_rn(q[j], sc), lo), xv[j0 + j]);
                        sum = __fadd_rn(sum, __fmul_rn(d, d));
                    }
                }
                const float err = __fdiv_rn(sum, (float)GROUP);
                if (mine && (first || err < best_err)) { best_err = err; best_lo = lo; best_sc = sc; }
                if (mine) first = false;
            }
            const float best_rs = __builtin_amdgcn_rcpf(best_sc);
#pragma unroll
            for (int j0 = 0; j0 < GROUP; j0 += 8) {
                float q[8];
                sk_codes8(xv + j0, q, best_lo, best_sc, best_rs, levels, tie);
#pragma unroll
                for (int j = 0; j < 8; ++j) p[j0 + j] = __fadd_rn(__fmul_rn(q[j], best_sc), best_lo);
            }
        } else {
        float mn = p[0], mx = p[0];
        for (int j = 1; j < group; ++j) { mn = fminf(mn, p[j]); mx = fmaxf(mx, p[j]); }
        const float mid = __fmul_rn(__fadd_rn(mx, mn), 0.5f), rng = __fsub_rn(mx, mn);
        float best_err = 0.f, best_lo = 0.f, best_sc = 1.f;
        for (int k = 0; k < al.n; ++k) {
            const float ar = __fmul_rn(al.a[k], rng);
            const float lo = __fsub_rn(mid, __fmul_rn(ar, 0.5f));
            const float sc = fmaxf(__fdiv_rn(ar, levels), 1e-8f);
            const float rs = __builtin_amdgcn_rcpf(sc);
            float sum = 0.f;
            for (int j = 0; j < group; ++j) {
                const float q = sk_code(p[j], lo, sc, rs, levels);
                const float d = __fsub_rn(__fadd_rn(__fmul_rn(q, sc), lo), p[j]);
                sum = __fadd_rn(sum, __fmul_rn(d, d));
            }
            const float err = __fdiv_rn(sum, (float)group);
            if (k == 0 || err < best_err) { best_err = err; best_lo = lo; best_sc = sc; }
        }
        const float best_rs = __builtin_amdgcn_rcpf(best_sc);
        for (int j = 0; j < group; ++j) {
            const float q = sk_code(p[j], best_lo, best_sc, best_rs, levels);
            p[j] = __fadd_rn(__fmul_rn(q, best_sc), best_lo);
        }
        }
    }
    __syncthreads();

    if constexpr (ERR) {
        // `place` names the words of channels (without `inv`: of places in the order); looking the order up again for each row
        // cost 2.9 of 22.5 us
        const bool staged = scatter || !perm;
        for (int lr = lr_base; lr < rows_pb && lr_base < rpp; lr += rpp) {
            if (row0 + lr >= n_rows) continue;
            const Where w = where(lr);
            const T *src = x + (int64_t)w.bh * x_stride_bh + (int64_t)w.t * D;
            const int32_t *iv = inv ? inv + (int64_t)w.head * D : nullptr;
            const float *srcl = s_x + lr * G * gstride;
            double sum = 0.0;
            for (int c0 = cq * 8; c0 < (int)D; c0 += tpr * 8) {
                float v[8];
                if (vec) Vec8<T>::ld(src + c0, v);
                if (staged) place(w.head, c0);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int c = c0 + k;
                    if (c >= (int)D) continue;
                    const double d = (double)__fsub_rn(srcl[staged ? off[k] : pos(iv ? iv[c] : c)], vec ? v[k] : Elem<T>::ld(src + c));
                    sum += d * d;
                }
            }
            err[((int64_t)(2 * blockIdx.z + blockIdx.y) * n_rows + row0 + lr) * tpr + cq] = sum;
        }
        return;
    }
    for (int lr = lr_base; lr < rows_pb && lr_base < rpp; lr += rpp) {
        if (row0 + lr >= n_rows) continue;
        const Where w = where(lr);
        T *dst = out + (int64_t)w.bh * out_stride_bh + (int64_t)w.t * D;
        const int32_t *pm = perm ? perm + (int64_t)w.head * D : nullptr;
        const float *srcl = s_x + lr * G * gstride;
        for (int c0 = cq * 8; c0 < (int)D; c0 += tpr * 8) {
            float v[8];
            place(w.head, c0);
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = c0 + k < (int)D ? srcl[off[k]] : 0.f;
            if (vec) {
                Vec8<T>::st(dst + c0, v);
            } else {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (c0 + k < (int)D) Elem<T>::st(dst + (pm ? pm[c0 + k] : c0 + k), v[k]);
            }
        }
    }
}

// ---- channel orders of the first flushed chunk (veloxquant_mlx/cache/skvq_cache.py:186-224) ----
//
// Three launches for keys and values together (they take different blocks of the same launches: latency is what they
// cost, and one after the other they took 105 us instead of 53): the candidate order of every head (channels by their range over the chunk's rows, equal
// ranges in channel order), the squared round-trip error of the stored and of the candidate order (the ERR form of the
// kernel above), and the choice per head (the candidate only where its mean error is lower).  Latency is all there is
// to them: 8 x 8 heads of 123 rows of 128 channels took 0.21 ms a tensor as library reductions and sorts.
constexpr int SK_ORD_THREADS = 1024;

// floats as unsigned numbers in the same order (NaNs are kept apart)
__device__ __forceinline__ uint32_t sk_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
}
__device__ __forceinline__ float sk_unkey(uint32_t k) { return __uint_as_float(k & 0x80000000u ? k & 0x7fffffffu : ~k); }

// One block per head; W channels (8 where rows move as 16-byte pieces, else 1) a thread, so that the block reads
// SK_ORD_THREADS / (D / W) rows at a time.  LDS: smallest, largest, NaN mark of every channel, then ranges and places; channel c's
// words lie at slot(c), piece after piece for equal c % W, so that the pieces of a wave meet different banks.
// Few blocks, so a block's own instructions are what it waits for (8 heads of 8 x 123 rows of 128 channels, two tensors: 26.8 -> 15.2 us): two
// rows an operation and one comparison for a NaN in either (eight operations a value and row before, now two and a half), up to
// AHEAD rows requested at once, the lanes of a wave with the same channels reduced before the LDS atomics, and
// SK_ORD_THREADS / D threads to a channel's comparisons (128 in a row by an eighth of the threads before).

// smallest and largest of the two halves (rows) of a wave, in every lane
template <int HALF> __device__ __forceinline__ void sk_fold_lanes(float &mn, float &mx, uint32_t &nan) {
    mn = fminf(mn, __shfl_xor(mn, HALF));
    mx = fmaxf(mx, __shfl_xor(mx, HALF));
    nan |= __shfl_xor(nan, HALF);
}
template <typename T, int W>
__global__ __launch_bounds__(SK_ORD_THREADS)
void skvq_order_kernel(SkSides sides, int64_t B, int64_t H, int64_t r, int D, int64_t x_stride_bh) {
    const T *__restrict__ x = (const T *)sides.t[blockIdx.z].x;
    int32_t *__restrict__ perm = sides.t[blockIdx.z].perm, *__restrict__ inv = sides.t[blockIdx.z].inv;
    constexpr int AHEAD = W == 8 ? 16 / (int)sizeof(T) : 16;   // (twice as many pieces of 16 bytes spill)
    extern __shared__ uint32_t s_ord[];
    uint32_t *s_mn = s_ord, *s_mx = s_ord + D, *s_nan = s_ord + 2 * D;
    float *s_rng = reinterpret_cast<float *>(s_ord);
    int32_t *s_place = reinterpret_cast<int32_t *>(s_ord + D);
    const int tid = threadIdx.x;
    const int64_t h = blockIdx.x, n = B * r;
    for (int c = tid; c < D; c += SK_ORD_THREADS) { s_mn[c] = ~0u; s_mx[c] = 0u; s_nan[c] = 0u; }
    __syncthreads();
    const int pieces = D / W, width = pieces < SK_ORD_THREADS ? pieces : SK_ORD_THREADS, rows = SK_ORD_THREADS / width;
    auto slot = [&](int c) { return W == 1 ? c : c % W * pieces + c / W; };
    const int p0 = tid % width, row0 = tid / width;
    // a wave holds whole rows, and the number of its lanes between equal channels is a power of two
    const bool fold = width < 64 && 64 % width == 0;
    for (int p = p0; p < pieces && row0 < rows; p += width) {
        float mn[W], mx[W];
        bool bad[W];
#pragma unroll
        for (int k = 0; k < W; ++k) { mn[k] = INFINITY; mx[k] = -INFINITY; bad[k] = false; }
        int b = row0 / (int)r, t = row0 - b * (int)r;   // the thread's next row, carried along: no division in the loop
#pragma unroll 1
        for (int64_t i = row0; i < n; i += AHEAD * rows) {
            typename Vec8<T>::Raw raw[AHEAD];
            float one[AHEAD];
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {   // past the end the last row comes again
                const T *src = x + (b * H + h) * x_stride_bh + (int64_t)t * D + (int64_t)p * W;
                if constexpr (W == 8) raw[j] = Vec8<T>::request(src);
                else one[j] = Elem<T>::ld(src);
                if (i + (j + 1) * rows < n)
                    for (t += rows; t >= (int)r; t -= (int)r) ++b;
            }
#pragma unroll
            for (int j = 0; j < AHEAD; j += 2) {   // two rows an operation: min3, max3, one comparison for a NaN in either
                float v[8], u[8];
                if constexpr (W == 8) {
                    Vec8<T>::unpack(raw[j], v);
                    Vec8<T>::unpack(raw[j + 1], u);
                } else {
                    v[0] = one[j];
                    u[0] = one[j + 1];
                }
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    mn[k] = fminf(fminf(mn[k], v[k]), u[k]);
                    mx[k] = fmaxf(fmaxf(mx[k], v[k]), u[k]);
                    bad[k] = bad[k] | (bool)__builtin_isunordered(v[k], u[k]);
                }
            }
        }
        uint32_t nan = 0u;
#pragma unroll
        for (int k = 0; k < W; ++k) nan |= bad[k] ? 1u << k : 0u;
        if (fold) {   // (one pass of the loop over p, every lane in it)
#pragma unroll
            for (int k = 0; k < W; ++k) {
                uint32_t none = 0u, &mark = k == 0 ? nan : none;
                if (width <= 32) sk_fold_lanes<32>(mn[k], mx[k], mark);
                if (width <= 16) sk_fold_lanes<16>(mn[k], mx[k], mark);
                if (width <= 8) sk_fold_lanes<8>(mn[k], mx[k], mark);
            }
        }
        if (fold && (tid & 63) >= (width < 8 ? 8 : width)) continue;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            atomicMin(&s_mn[k * (W == 1 ? 0 : pieces) + p], sk_key(mn[k]));
            atomicMax(&s_mx[k * (W == 1 ? 0 : pieces) + p], sk_key(mx[k]));
            if (nan >> k & 1u) s_nan[k * (W == 1 ? 0 : pieces) + p] = 1u;
        }
    }
    __syncthreads();
    for (int c = tid; c < D; c += SK_ORD_THREADS) {   // each thread its own words: range and place take the values' place
        s_rng[c] = s_nan[c] ? NAN : __fsub_rn(sk_unkey(s_mx[c]), sk_unkey(s_mn[c]));
        s_place[c] = 0;
    }
    __syncthreads();
    // place = channels before this one; a NaN comes after every number.  `share` threads a channel, a run of the others each.
    const int share = D < SK_ORD_THREADS ? SK_ORD_THREADS / D : 1, run = (D + share - 1) / share;
    const int part = D < SK_ORD_THREADS ? tid / D : 0;
    for (int c = D < SK_ORD_THREADS ? tid % D : tid; c < D && part < share; c += SK_ORD_THREADS) {
        const float mine = s_rng[slot(c)];
        const bool mine_nan = mine != mine;
        const int to = (part + 1) * run < D ? (part + 1) * run : D;
        int place = 0;
#pragma unroll 8
        for (int j = part * run; j < to; ++j) {
            const float o = s_rng[slot(j)];
            const bool o_nan = o != o;
            const bool before = mine_nan ? !o_nan : o < mine, same = mine_nan ? o_nan : o == mine;
            place += (before || (same && j < c)) ? 1 : 0;
        }
        atomicAdd(&s_place[slot(c)], place);
    }
    __syncthreads();
    for (int c = tid; c < D; c += SK_ORD_THREADS) {
        const int place = s_place[slot(c)];
        perm[h * D + place] = c;
        inv[h * D + c] = place;
    }
}

// One block per head: both orders' errors summed in one fixed order, and the head's order kept or replaced by the stored one.
__global__ __launch_bounds__(SK_ORD_THREADS)
void skvq_choose_kernel(const double *__restrict__ err, int64_t B, int64_t H, int64_t r, int tpr, int D, SkSides sides) {
    int32_t *__restrict__ perm = sides.t[blockIdx.z].perm, *__restrict__ inv = sides.t[blockIdx.z].inv;
    err += (int64_t)blockIdx.z * 2 * B * H * r * tpr;
    __shared__ double s_sum[2][SK_ORD_THREADS];
    const int tid = threadIdx.x;
    const int64_t h = blockIdx.x, n_rows = B * H * r, per_bh = r * tpr;
    double a[2] = {0.0, 0.0};
    int64_t b = tid / per_bh, i = tid - b * per_bh;   // the errors of the head, sequence after sequence
    const double *e = err + h * per_bh, *e1 = e + n_rows * tpr;
    const int64_t step = H * per_bh;
#pragma unroll 8
    for (int64_t n = tid; n < B * per_bh; n += SK_ORD_THREADS) {
        a[0] += e[b * step + i];
        a[1] += e1[b * step + i];
        for (i += SK_ORD_THREADS; i >= per_bh; i -= per_bh) ++b;
    }
    s_sum[0][tid] = a[0];
    s_sum[1][tid] = a[1];
    for (int w = SK_ORD_THREADS / 2; w > 0; w >>= 1) {
        __syncthreads();
        if (tid < w) { s_sum[0][tid] += s_sum[0][tid + w]; s_sum[1][tid] += s_sum[1][tid + w]; }
    }
    __syncthreads();
    const double count = (double)(B * r * D);
    if (s_sum[1][0] / count < s_sum[0][0] / count) return;   // (an error that is not a number keeps the stored order)
    for (int c = tid; c < D; c += SK_ORD_THREADS) perm[h * D + c] = inv[h * D + c] = c;
}

// how a round-trip launch covers its rows
struct SkPlan {
    int threads, tpr;
    int64_t G, rows_pb, n_rows, blocks;
    uint64_t group_magic;
    size_t lds;
};
static int plan_skvq(const char *fn, int64_t B, int64_t H, int64_t r, int64_t D, int bits, int group, const float *alphas, int n_alphas,
                     SkPlan &p, SkAlphas &al) {
    VQ_REQUIRE(bits >= 1 && bits <= 8, VQ_ERR_INVALID, "%s: bits must be in [1, 8], got %d", fn, bits);
    VQ_REQUIRE(group >= 1, VQ_ERR_INVALID, "%s: group_size must be >= 1, got %d", fn, group);
    VQ_REQUIRE(alphas && n_alphas >= 1 && n_alphas <= SK_MAX_ALPHAS, VQ_ERR_INVALID,
               "%s: between 1 and %d clip factors, got %d", fn, SK_MAX_ALPHAS, n_alphas);
    for (int k = 0; k < n_alphas; ++k)
        VQ_REQUIRE(alphas[k] > 0.f && alphas[k] <= 1.f, VQ_ERR_INVALID, "%s: alphas must lie in (0, 1], got %g", fn,
                   (double)alphas[k]);
    VQ_REQUIRE(B >= 0 && H >= 0 && r >= 0 && D >= 0, VQ_ERR_INVALID, "%s: negative dimension", fn);
    al.n = n_alphas;
    for (int k = 0; k < SK_MAX_ALPHAS; ++k) al.a[k] = k < n_alphas ? alphas[k] : 1.f;
    p.G = (D + group - 1) / group;
    const int64_t row_words = p.G * (group + 1);
    VQ_REQUIRE(p.G <= SK_THREADS && row_words * 4 <= 48 * 1024 && group < 65536, VQ_ERR_UNSUPPORTED,
               "%s: head_dim %lld with group %d does not fit a block (at most %d groups, 48 KB per row)", fn,
               (long long)D, group, SK_THREADS);
    if (B * H * r * D == 0) return VQ_OK;
    // one wave per block where a wave covers whole rows: blocks then interleave freely on a CU (the
    // phases of a block do not overlap each other, those of different blocks do)
    p.threads = (p.G <= 64 && (p.G * group + 7) / 8 <= 64) ? 64 : SK_THREADS;
    p.rows_pb = p.threads / p.G;
    if (p.rows_pb * row_words * 4 > 48 * 1024) p.rows_pb = 48 * 1024 / (row_words * 4);
    p.n_rows = B * H * r;
    p.blocks = (p.n_rows + p.rows_pb - 1) / p.rows_pb;
    VQ_REQUIRE(p.n_rows <= 0x7fffffff, VQ_ERR_UNSUPPORTED, "%s: too many rows (%lld)", fn, (long long)p.n_rows);
    // floor(j / group) == (j * magic) >> 32 for j, group < 2^16 (a row holds at most 12288 words in LDS)
    p.group_magic = (1ull << 32) / (uint64_t)group + 1;
    const int64_t pieces = (p.G * group + 7) / 8;   // threads side by side on a row (eight channels each)
    p.tpr = (int)(pieces < p.threads ? pieces : p.threads);
    p.lds = (size_t)(p.rows_pb * row_words * 4);
    return VQ_OK;
}

template <typename T, bool ERR>
static void launch_skvq(const SkPlan &p, const SkAlphas &al, const SkSides &sides, int tensors, double *err, int64_t B, int64_t H, int64_t r,
                        int64_t D, int64_t xs, int64_t os, int group, bool vec, hipStream_t st) {
    const dim3 grid((unsigned)p.blocks, ERR ? 2 : 1, (unsigned)tensors);
#define VQ_SK_LAUNCH(GROUP)                                                                                                   \
    hipLaunchKernelGGL((skvq_roundtrip_kernel<T, GROUP, ERR>), grid, dim3(p.threads), p.lds, st, sides, err, B * H, H, r, D, xs, os, \
                       group, p.group_magic, (int)p.G, (int)p.rows_pb, p.tpr, vec, al)
    if (group == 32) VQ_SK_LAUNCH(32);
    else if (group == 64) VQ_SK_LAUNCH(64);
    else VQ_SK_LAUNCH(0);
#undef VQ_SK_LAUNCH
}

}  // namespace vq

using namespace vq;

extern "C" int vq_skvq_clipped_roundtrip(const void *x, void *out, int dtype, int64_t B, int64_t H, int64_t r,
                                         int64_t D, int64_t x_stride_bh, int64_t out_stride_bh, const int32_t *perm,
                                         const int32_t *inv, int bits, int group, const float *alphas, int n_alphas, void *stream) {
    const char *fn = "vq_skvq_clipped_roundtrip";
    SkPlan p;
    SkAlphas al;
    VQ_REQUIRE(is_float_tag(dtype), VQ_ERR_INVALID, "%s: unsupported dtype tag %d", fn, dtype);
    const int rc = plan_skvq(fn, B, H, r, D, bits, group, alphas, n_alphas, p, al);
    if (rc != VQ_OK) return rc;
    if (B * H * r * D == 0) return VQ_OK;
    VQ_REQUIRE(x && out, VQ_ERR_INVALID, "%s: null pointer", fn);
    VQ_REQUIRE(x_stride_bh >= r * D && out_stride_bh >= r * D, VQ_ERR_INVALID, "%s: stride below r * D", fn);
    VQ_REQUIRE(perm || !inv, VQ_ERR_INVALID, "%s: inv given without perm", fn);
    // whether rows can move as 16-byte pieces
    const bool vec = (perm == nullptr || inv != nullptr) && D % 8 == 0 && x_stride_bh % 8 == 0 && out_stride_bh % 8 == 0 &&
                     ((uintptr_t)x % 16 == 0) && ((uintptr_t)out % 16 == 0);
    SkSides sides = {};
    sides.t[0] = {x, out, (int32_t *)perm, (int32_t *)inv, (float)((1 << bits) - 1)};
    VQ_DISPATCH_FLOAT(dtype, T, {
        launch_skvq<T, false>(p, al, sides, 1, nullptr, B, H, r, D, x_stride_bh, out_stride_bh, group, vec, (hipStream_t)stream);
    })
    VQ_HIP_CHECK_LAUNCH(fn);
    return VQ_OK;
}

extern "C" size_t vq_skvq_channel_orders_workspace(int64_t B, int64_t H, int64_t r, int64_t D, int group, int tensors) {
    if (B < 1 || H < 1 || r < 1 || D < 1 || group < 1 || tensors < 1 || tensors > 2) return 0;
    const int64_t pieces = ((D + group - 1) / group * group + 7) / 8, tpr = pieces < SK_THREADS ? pieces : SK_THREADS;
    return (size_t)(2 * tensors * B * H * r * tpr) * sizeof(double);
}

extern "C" int vq_skvq_channel_orders(const void *x, const void *x2, int dtype, int64_t B, int64_t H, int64_t r, int64_t D, int64_t x_stride_bh,
                                      int bits, int bits2, int group, const float *alphas, int n_alphas, int32_t *perm, int32_t *inv,
                                      void *workspace, size_t workspace_bytes, void *stream) {
    const char *fn = "vq_skvq_channel_orders";
    SkPlan p;
    SkAlphas al;
    const int tensors = x2 != nullptr ? 2 : 1;
    VQ_REQUIRE(is_float_tag(dtype), VQ_ERR_INVALID, "%s: unsupported dtype tag %d", fn, dtype);
    VQ_REQUIRE(B >= 1 && H >= 1 && r >= 1 && D >= 1, VQ_ERR_INVALID, "%s: empty chunk", fn);
    const int rc = plan_skvq(fn, B, H, r, D, bits, group, alphas, n_alphas, p, al);
    if (rc != VQ_OK) return rc;
    VQ_REQUIRE(x2 == nullptr || (bits2 >= 1 && bits2 <= 8), VQ_ERR_INVALID, "%s: bits must be in [1, 8], got %d", fn, bits2);
    VQ_REQUIRE(x && perm && inv && workspace, VQ_ERR_INVALID, "%s: null pointer", fn);
    VQ_REQUIRE(x_stride_bh >= r * D, VQ_ERR_INVALID, "%s: stride below r * D", fn);
    VQ_REQUIRE(H <= 0x7fffffff, VQ_ERR_UNSUPPORTED, "%s: too many heads", fn);
    VQ_REQUIRE(workspace_bytes >= vq_skvq_channel_orders_workspace(B, H, r, D, group, tensors), VQ_ERR_WORKSPACE, "%s: workspace too small", fn);
    const bool vec = D % 8 == 0 && x_stride_bh % 8 == 0 && (((uintptr_t)x | (uintptr_t)x2) & 15u) == 0;
    double *err = (double *)workspace;
    hipStream_t st = (hipStream_t)stream;
    SkSides sides = {};
    sides.t[0] = {x, nullptr, perm, inv, (float)((1 << bits) - 1)};
    if (x2 != nullptr) sides.t[1] = {x2, nullptr, perm + H * D, inv + H * D, (float)((1 << bits2) - 1)};
    const dim3 heads((unsigned)H, 1, (unsigned)tensors);
    VQ_DISPATCH_FLOAT(dtype, T, {
        const size_t lds = (size_t)D * 12;   // D <= 12288 words of a row, so at most 144 KB
        auto kernel = vec ? skvq_order_kernel<T, 8> : skvq_order_kernel<T, 1>;
        if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        hipLaunchKernelGGL(kernel, heads, dim3(SK_ORD_THREADS), lds, st, sides, B, H, r, (int)D, x_stride_bh);
        launch_skvq<T, true>(p, al, sides, tensors, err, B, H, r, D, x_stride_bh, x_stride_bh, group, vec, st);
    })
    hipLaunchKernelGGL(skvq_choose_kernel, heads, dim3(SK_ORD_THREADS), 0, st, err, B, H, r, p.tpr, (int)D, sides);
    VQ_HIP_CHECK_LAUNCH(fn);
    return VQ_OK;
}
