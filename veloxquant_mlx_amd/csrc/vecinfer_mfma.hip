// VecInfer nearest-centroid assignment on the matrix unit (gfx950, wave64), with indices
// identical to the sequential float32 rule of veloxquant_mlx/metal/src/vecinfer_quantize.metal:8-28
// (squares rounded separately, dimensions added left to right, strict '<').
//
// The matrix unit cannot reproduce that rounding order, so it only names the few centroids that can win,
// and the exact rule chooses among them:
//
//   d2[c, v] = |c|^2 - 2 c.v + |v|^2   v_mfma_f32_32x32x16_f16, 32 centroids x 32 sub-vectors a product.  c and v
//       travel as fp16 high part + fp16 remainder, |c|^2 and |v|^2 as two fp16 parts in k-slots of their own, so the
//       accumulator input is the constant zero.  Codebook and sub-vectors are first multiplied by one power of two that
//       puts max|c|^2 in [256, 1024) (remainders stay out of the subnormals); d2 is then good to 2^-19 (|c|^2 + |v|^2), apart from
//       an error of |v|^2 that all scores of a sub-vector share: 3 2^-22 from the parts of c and v and the product of remainders
//       that is left out, 2^-22 from those of |c|^2, 2^-21 from the accumulation, whose rounding the unit does not
//       document.  That last part is measured: over 5 x 10^5 scores each of normal, equal, near, very long, all-mantissa-bits, fp16
//       half-way, wide-exponent and one-large-channel vectors the accumulation is off by 2^-21.5 at most (beyond the constant
//       margin's reach), and twice the largest error of a score is 13 % of the margin below without its tag bits.
//   A *cell* is the 16 scores one lane holds of a product: 16 centroids, one sub-vector.  |v|^2 carries a small surplus
//       that keeps every score positive, so float bits order as integers: the smallest of a cell costs eight min3, the
//       tile number goes into its seven low bits (one and-or), and the two smallest cells of the lane are kept in two
//       more operations: 11 vector operations for 16 scores (0.69 a score; tracking the two smallest scores
//       themselves with their positions took 2.5).
//   If the second cell is farther than eps (2^-16 |v|^2 + 2^-14 d2: filter error of both sides, |c|^2 <= 2 |v|^2 + 2 d2, plus the tag bits) the
//       exact rule runs over the 16 centroids of the first; else, if both leaders come from different lanes and nothing
//       else lies within eps, over the 32 of both; else over the whole codebook (rare: a wave does it together).
//
// Two forms.  IMAGE: the block builds the codebook once in LDS as operand tiles (24 bytes a centroid of four dimensions,
// 48 of eight) and its waves walk all tiles for 64 sub-vectors at a time; four waves a SIMD, because a
// product keeps the vector unit waiting for its 16 results.  SPLIT, for few sub-vectors: a block takes 64 sub-vectors and
// its waves share out the *tiles*, straight from memory; their cells are merged through LDS and the exact rule runs
// with one lane a centroid.  SPLIT spends twice the vector work a sub-vector (every wave forms its operands from float
// rows) but fills the chip from a few dozen blocks on.  Where the line lies: see kSplitMax.
#include <atomic>
#include <type_traits>

#include "vecinfer.hpp"

namespace vq {

typedef uint32_t u32;
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int VM_MAXC = 4096;   // tile numbers have seven bits
// SPLIT up to this many sub-vectors and above kSplitC centroids: two rounds of its blocks (one to a CU).  Measured, us a call,
// SPLIT / IMAGE: 4096 centroids of four dimensions, 512 sub-vectors 9.9 / 19.3, 16384 10.7 / 27.5, 65536 42 / 26.6; 2048 of
// eight 9.8 / 18.0, 9.5 / 21.3, 38 / 24.0; 1024 of four 8.1 / 8.1, 8.1 / 9.2, 26.9 / 12.3.
constexpr int64_t kSplitMax = 32768;
constexpr int kSplitC = 1024;
// codebooks up to this size track quarter cells (seven bits: 16 tiles and four runs, with room)
constexpr int kFineC = 512;

__device__ __forceinline__ u32 umin3(u32 a, u32 b, u32 c) { return min(min(a, b), c); }
__device__ __forceinline__ u32 umed3(u32 a, u32 b, u32 c) {
    u32 d;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}
// the smallest of a lane's 16 scores of a product, with the tile number in its low bits
__device__ __forceinline__ u32 cell_key(const f32x16 &d, u32 mask, int tile) {
    u32 s[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = __float_as_uint(d[i]);
    const u32 a = umin3(s[0], s[1], s[2]), b = umin3(s[3], s[4], s[5]), c = umin3(s[6], s[7], s[8]);
    const u32 e = umin3(s[9], s[10], s[11]), f = umin3(s[12], s[13], s[14]);
    const u32 m = min(umin3(a, b, c), umin3(e, f, s[15]));
    u32 r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(mask), "s"(tile));
    return r;
}
// The same at a quarter of the cell: the four runs of four scores apart, run number below the tile number.  Eighteen
// operations for 16 scores, but the exact rule then runs over four centroids: for small codebooks, where it is most of the work.
__device__ __forceinline__ void keep_quarters(u32 &k1, u32 &k2, const f32x16 &d, u32 mask, int tile) {
    u32 q[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const u32 a = __float_as_uint(d[4 * g]), b = __float_as_uint(d[4 * g + 1]), c = __float_as_uint(d[4 * g + 2]);
        const u32 m = min(umin3(a, b, c), __float_as_uint(d[4 * g + 3]));
        asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(q[g]) : "v"(m), "v"(mask), "s"(4 * tile + g));
    }
#pragma unroll
    for (int g = 0; g < 4; g += 2) {   // two new keys into the sorted pair
        const u32 m = umed3(k1, q[g], q[g + 1]);
        k1 = umin3(k1, q[g], q[g + 1]);
        k2 = min(k2, m);
    }
}
// a new key into the sorted pair k1 <= k2
__device__ __forceinline__ void keep_two(u32 &k1, u32 &k2, u32 key) {
    k2 = umed3(k1, k2, key);
    k1 = min(k1, key);
}
// lanes 0..31 of a with lanes 32..63 of b: a = [a.low, b.low], b = [a.high, b.high]
__device__ __forceinline__ void swap_halves(u32 &a, u32 &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// ---- the key transform in front of the assignment, and the reconstruction behind it --------
//
// With LT > 0 the sub-vectors are not taken as they are: 64 consecutive sub-vectors are 64 / LT
// whole tokens of D = LT * SUB channels (lane j of a group of LT lanes holds channels
// [SUB j, SUB (j + 1))), and each token first goes through  k~ = (k / smooth) @ H  with H the
// orthonormal Sylvester-Hadamard matrix (entries +-h in natural order), done as a fast
// Walsh-Hadamard transform across the LT lanes: in-lane butterflies over the SUB registers, then
// one butterfly per lane bit (cross-lane moves inside the row of 16, LDS permutes beyond it), then
// the scale h.  Optionally the chosen centroids go back the same way, k^ = (c @ H^T) * smooth
// (H is symmetric), and k~ itself can be written out.  This is the reference's fused key
// encode+decode (veloxquant_mlx/metal/_vecinfer.py:225-293) as a front and back end of the
// MFMA assignment.
struct KeyXform {
    const float *smooth;   // [smooth_rows, D] float32 or null
    int smooth_rows;       // 1 or the number of heads
    int64_t heads, S;      // keys are [B, heads, S, D]
    float h;               // |H[0][0]|
    void *k_hat;           // [N * SUB] reconstruction in dtype hat_dtype, or null
    int hat_dtype;
    float *k_tilde;        // [N * SUB] transformed keys, or null
};

template <int CTRL> __device__ __forceinline__ float xform_dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// value of lane (lane ^ M)
template <int M> __device__ __forceinline__ float lane_xor(float x) {
    if constexpr (M == 1) return xform_dpp<0xB1>(x);        // quad_perm [1,0,3,2]
    else if constexpr (M == 2) return xform_dpp<0x4E>(x);   // quad_perm [2,3,0,1]
    else if constexpr (M == 8) return xform_dpp<0x128>(x);  // row_ror 8
    else return __shfl_xor(x, M);
}
template <int SUB, int M> __device__ __forceinline__ void lane_butterfly(float (&x)[8], int lane) {
    const bool upper = (lane & M) != 0;
#pragma unroll
    for (int e = 0; e < SUB; ++e) {
        const float p = lane_xor<M>(x[e]);
        x[e] = upper ? p - x[e] : x[e] + p;
    }
}
// unnormalised Walsh-Hadamard transform of the LT * SUB values a group of LT lanes holds
template <int SUB, int LT> __device__ __forceinline__ void wht_lanes(float (&x)[8], int lane) {
#pragma unroll
    for (int hlf = 1; hlf < SUB; hlf <<= 1)
#pragma unroll
        for (int i = 0; i < SUB; i += 2 * hlf)
#pragma unroll
            for (int k = i; k < i + hlf; ++k) {
                const float a = x[k], b = x[k + hlf];
                x[k] = a + b;
                x[k + hlf] = a - b;
            }
    if constexpr (LT > 1) lane_butterfly<SUB, 1>(x, lane);
    if constexpr (LT > 2) lane_butterfly<SUB, 2>(x, lane);
    if constexpr (LT > 4) lane_butterfly<SUB, 4>(x, lane);
    if constexpr (LT > 8) lane_butterfly<SUB, 8>(x, lane);
    if constexpr (LT > 16) lane_butterfly<SUB, 16>(x, lane);
    if constexpr (LT > 32) lane_butterfly<SUB, 32>(x, lane);
}

// ---- rows of the codebook ---------------------------------------------------------------------

// N rows at once: every load is on its way before the first is used
template <int SUB, int N>
__device__ __forceinline__ void load_centroids(const void *cb, int ct, bool aligned, const int (&c)[N], float (&row)[N][SUB]) {
    if (!aligned) {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int e = 0; e < SUB; ++e) row[i][e] = ld_any(cb, ct, (int64_t)c[i] * SUB + e);
    } else if (ct == VQ_F32) {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int e = 0; e < SUB; e += 4) {
                const float4 v = *reinterpret_cast<const float4 *>((const float *)cb + (int64_t)c[i] * SUB + e);
                row[i][e] = v.x; row[i][e + 1] = v.y; row[i][e + 2] = v.z; row[i][e + 3] = v.w;
            }
    } else {
        u32 w[N][SUB / 2];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if constexpr (SUB == 8) {
                const uint4 v = *reinterpret_cast<const uint4 *>((const u16 *)cb + (int64_t)c[i] * 8);
                w[i][0] = v.x; w[i][1] = v.y; w[i][2] = v.z; w[i][3] = v.w;
            } else {
                const uint2 v = *reinterpret_cast<const uint2 *>((const u16 *)cb + (int64_t)c[i] * 4);
                w[i][0] = v.x; w[i][1] = v.y;
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int e = 0; e < SUB / 2; ++e) {
                const f16x2 h = __builtin_bit_cast(f16x2, w[i][e]);
                row[i][2 * e] = ct == VQ_F16 ? (float)h[0] : __uint_as_float(w[i][e] << 16);
                row[i][2 * e + 1] = ct == VQ_F16 ? (float)h[1] : __uint_as_float(w[i][e] & 0xffff0000u);
            }
    }
}
template <int SUB>
__device__ __forceinline__ void load_centroid(const void *cb, int ct, bool aligned, int c, float (&row)[SUB]) {
    const int cc[1] = {c};
    float r[1][SUB];
    load_centroids<SUB, 1>(cb, ct, aligned, cc, r);
#pragma unroll
    for (int e = 0; e < SUB; ++e) row[e] = r[0][e];
}
template <int SUB> __device__ __forceinline__ float norm2(const float *row) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < SUB; ++e) s = __builtin_fmaf(row[e], row[e], s);
    return s;
}
// the exact rule
template <int SUB> __device__ __forceinline__ float exact_dist(const float *x, const float *c) {
    float dist = 0.0f;
#pragma unroll
    for (int i = 0; i < SUB; ++i) {
        const float d = __fsub_rn(x[i], c[i]);
        dist = __fadd_rn(dist, __fmul_rn(d, d));
    }
    return dist;
}
// A float as fp16 high part and remainder.  The value is pinned first: left alone, the compiler forms the high part of a
// fused product once from the rounded float and once from the exact product, and at fp16 ties the two differ.
__device__ __forceinline__ u32 high_and_rest(float v) {
    asm("" : "+v"(v));
    const f16 h = (f16)v;
    return __builtin_bit_cast(u32, f16x2{h, (f16)(v - (float)h)});
}
__device__ __forceinline__ u32 pack_h2(float a, float b) { return __builtin_bit_cast(u32, f16x2{(f16)a, (f16)b}); }
// floats (products with powers of two: exact) as fp16 high parts and remainders, packed in pairs
template <int SUB> __device__ __forceinline__ void split_h(const float *v, u32 *hi, u32 *lo) {
#pragma unroll
    for (int e = 0; e < SUB; e += 2) {
        const f16 a = (f16)v[e], b = (f16)v[e + 1];
        hi[e / 2] = __builtin_bit_cast(u32, f16x2{a, b});
        lo[e / 2] = pack_h2(v[e] - (float)a, v[e + 1] - (float)b);
    }
}
// The power of two that puts cmax2 = max |c|^2 into [256, 1024).  Codebooks that none does this to: of squares near zero, whose
// scores all lie within the margin; of squares near infinity (a diverged centroid), whose other centroids the fp16 parts of
// |c|^2 cannot hold -- the scale is not a number then, so that no sub-vector is in the filter's range (make_operands) and the
// exact rule alone decides.
__device__ __forceinline__ float codebook_scale(float cmax2) {
    if (!(cmax2 > 1e-30f)) return 1.f;
    if (!(cmax2 < 1e30f)) return NAN;
    const int e = (int)((__float_as_uint(cmax2) >> 23) & 255u) - 127;   // 2^e <= cmax2 < 2^(e+1)
    const int k = (e - 8) >> 1;                                         // floor
    return __uint_as_float((u32)(127 - k) << 23);
}

// Operand image of a centroid, in words.  SUB 4: [remainder 4 | high 4 | |c|^2 parts, 2^15 2^15]; lanes 0..31 read words
// 0..3 against [high | high] of the sub-vector, lanes 32..63 words 2..5 against [remainder | 1 1 | |v|^2 2^-15 parts].
// SUB 8: [high 8][remainder 8][|c|^2 parts, 2^15 2^15, 0 0 0 0]: a first product of high and remainder against the
// sub-vector's high part, a second of high and the last block against [remainder | 1 1, |v|^2 2^-15 parts, 0 ..].
template <int SUB> constexpr int image_words() { return SUB == 4 ? 6 : 12; }
constexpr u32 kTwo15 = 0x78007800u;   // fp16 2^15, twice

template <int SUB> __device__ __forceinline__ void centroid_image(const float *row, float cs, u32 *img) {
    float s[SUB], c2 = 0.f;
#pragma unroll
    for (int e = 0; e < SUB; ++e) {
        const float t = row[e] * cs;
        c2 = __builtin_fmaf(t, t, c2);
        s[e] = -2.f * t;
    }
    u32 hi[SUB / 2], lo[SUB / 2];
    split_h<SUB>(s, hi, lo);
    const u32 cc = high_and_rest(c2);
    if constexpr (SUB == 4) {
        img[0] = lo[0]; img[1] = lo[1]; img[2] = hi[0]; img[3] = hi[1]; img[4] = cc; img[5] = kTwo15;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) { img[e] = hi[e]; img[4 + e] = lo[e]; }
        img[8] = cc; img[9] = kTwo15; img[10] = 0; img[11] = 0;
    }
}

// A row past the end of the codebook: zeros for c, twice 65504 for |c|^2 and 65504 for the factors of |v|^2's parts, so its score
// 131008 + 2 |v|^2 lies above (32 + |v|)^2, the largest a centroid can have, by more than the margin for every |v| in
// the filter's range.  It never leads a cell that holds a centroid and never counts as near (the last centroid in its place, again and
// again, was as near as itself wherever it won, and sent one sub-vector in nc through the whole codebook: 16 centroids of four
// over 1048576 76 us, 14 since).
template <int SUB> __device__ __forceinline__ void pad_image(u32 *img) {
#pragma unroll
    for (int e = 0; e < image_words<SUB>(); ++e) img[e] = 0;
    img[SUB == 4 ? 4 : 8] = img[SUB == 4 ? 5 : 9] = 0x7bff7bffu;
}

// ---- sub-vectors -----------------------------------------------------------------------------

// One lane's sub-vector and the operands of the wave's 64: column block b holds sub-vectors 32 b + (lane & 31).
template <int SUB> struct SubVec {
    float xf[SUB];
    float sm[SUB];
    float x2;      // |v|^2, scaled
    bool far;      // out of the filter's range (NaN, infinities, far outside the codebook): the exact rule alone
    f16x8 B1[2], B2[2];
};

__device__ __forceinline__ f16x8 h8(u32 a, u32 b, u32 c, u32 d) { return __builtin_bit_cast(f16x8, make_uint4(a, b, c, d)); }

template <int SUB>
__device__ __forceinline__ uint4 load_raw(const void *x, int xt, int64_t sv, bool live) {
    uint4 r = make_uint4(0, 0, 0, 0);
    if (!live || xt == VQ_F32) return r;
    if constexpr (SUB == 8) r = *reinterpret_cast<const uint4 *>((const u16 *)x + sv * 8);
    else { const uint2 t = *reinterpret_cast<const uint2 *>((const u16 *)x + sv * 4); r.x = t.x; r.y = t.y; }
    return r;
}

template <int SUB, int LT>
__device__ __forceinline__ void take_subvec(SubVec<SUB> &s, const void *x, int xt, uint4 raw, int64_t sv, bool live, int lane,
                                            const KeyXform &kx) {
    float xf[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) xf[e] = 0.f;
    if (xt != VQ_F32) {
        const u32 w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int e = 0; e < SUB / 2; ++e) {
            if (xt == VQ_F16) {
                const f16x2 h = __builtin_bit_cast(f16x2, w[e]);
                xf[2 * e] = (float)h[0]; xf[2 * e + 1] = (float)h[1];
            } else {
                xf[2 * e] = __uint_as_float(w[e] << 16); xf[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
            }
        }
    } else if (live) {
#pragma unroll
        for (int e = 0; e < SUB; ++e) xf[e] = ((const float *)x)[sv * SUB + e];
    }
    if constexpr (LT > 0) {
        // the lane's channels of its token: divide by the smoothing factors, transform, scale
#pragma unroll
        for (int e = 0; e < SUB; ++e) s.sm[e] = 1.f;
        if (kx.smooth != nullptr && live) {
            const u32 token = (u32)(sv / LT);
            const u32 srow = kx.smooth_rows > 1 ? (token / (u32)kx.S) % (u32)kx.heads : 0;
            const float *sp = kx.smooth + ((int64_t)srow * LT + (lane & (LT - 1))) * SUB;
#pragma unroll
            for (int e = 0; e < SUB; ++e) { s.sm[e] = sp[e]; xf[e] = xf[e] / s.sm[e]; }
        }
        wht_lanes<SUB, LT>(xf, lane);
#pragma unroll
        for (int e = 0; e < SUB; ++e) xf[e] *= kx.h;
    }
#pragma unroll
    for (int e = 0; e < SUB; ++e) s.xf[e] = xf[e];
}

template <int SUB> __device__ __forceinline__ void make_operands(SubVec<SUB> &s, float cs) {
    float v[SUB];
    s.x2 = 0.f;
#pragma unroll
    for (int e = 0; e < SUB; ++e) {
        v[e] = s.xf[e] * cs;
        s.x2 = __builtin_fmaf(v[e], v[e], s.x2);
    }
    s.far = !(s.x2 <= 6.7e7f);   // 256 to 512 times the largest centroid; a NaN, of the sub-vector or of the scale, ends here too
    if (s.far) {
        s.x2 = 0.f;
#pragma unroll
        for (int e = 0; e < SUB; ++e) v[e] = 0.f;
    }
    // |v|^2 and the surplus that keeps every score positive: above the filter's error and the rounding of the two parts
    const float vv = __builtin_fmaf(s.x2, 1.52587890625e-05f, s.x2 + 0.03125f) * 3.0517578125e-05f;
    u32 hi[SUB / 2], lo[SUB / 2];
    split_h<SUB>(v, hi, lo);
    u32 ones = 0x3c003c00u, parts = high_and_rest(vv);
    if constexpr (SUB == 4) {
        u32 a0 = hi[0], a1 = hi[1], a2 = hi[0], a3 = hi[1];
        u32 b0 = lo[0], b1 = lo[1], b2 = ones, b3 = parts;
        swap_halves(a0, b0); swap_halves(a1, b1); swap_halves(a2, b2); swap_halves(a3, b3);
        s.B1[0] = h8(a0, a1, a2, a3);
        s.B1[1] = h8(b0, b1, b2, b3);
    } else {
        u32 a[4], b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) { a[e] = hi[e]; b[e] = hi[e]; swap_halves(a[e], b[e]); }
        s.B1[0] = h8(a[0], a[1], a[2], a[3]);
        s.B1[1] = h8(b[0], b[1], b[2], b[3]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a[e] = lo[e];
            b[e] = e == 0 ? ones : e == 1 ? parts : 0u;
            swap_halves(a[e], b[e]);
        }
        s.B2[0] = h8(a[0], a[1], a[2], a[3]);
        s.B2[1] = h8(b[0], b[1], b[2], b[3]);
    }
}

template <int SUB> __device__ __forceinline__ float margin(const SubVec<SUB> &s, u32 f1) {
    return __builtin_fmaf(6.103515625e-05f, __uint_as_float(f1), __builtin_fmaf(1.52587890625e-05f, s.x2, 2.44140625e-04f));
}
// first centroid of a cell's run g: a lane holds four runs of four rows of its tile
__device__ __forceinline__ int cell_centroid(u32 key, int half, int g) { return (int)(key & 127u) * 32 + 8 * g + 4 * half; }

__device__ __forceinline__ void take_nearer(float &d, int &i, float od, int oi) {
    if (od < d || (od == d && oi < i)) { d = od; i = oi; }
}
// The whole codebook by the exact rule for the sub-vectors of the lanes in `m`, one after the other by the whole wave:
// `x` is the lane's sub-vector, `my_idx` its result.
template <int SUB>
__device__ __forceinline__ void scan_all(unsigned long long m, const float (&x)[SUB], const void *cb, int ct, bool aligned, int nc, int lane,
                                         int &my_idx) {
    constexpr int N = SUB == 4 ? 8 : 2;   // rows in flight: more would spill
    while (m != 0) {
        const int src = __builtin_ctzll(m);
        m &= m - 1;
        float xs[SUB], d = INFINITY;
        int i = 0;   // (no distance below infinity: index 0)
#pragma unroll
        for (int e = 0; e < SUB; ++e) xs[e] = __shfl(x[e], src);
#pragma unroll 1
        for (int c0 = lane; c0 < nc; c0 += 64 * N) {
            int c[N];
            float row[N][SUB];
#pragma unroll
            for (int r = 0; r < N; ++r) c[r] = min(c0 + 64 * r, nc - 1);
            load_centroids<SUB, N>(cb, ct, aligned, c, row);
#pragma unroll
            for (int r = 0; r < N; ++r) {
                const float t = exact_dist<SUB>(xs, row[r]);
                if (t < d) { d = t; i = c[r]; }
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) take_nearer(d, i, __shfl_xor(d, o), __shfl_xor(i, o));
        if (lane == src) my_idx = i;
    }
}


template <int SUB, int LT>
__device__ __forceinline__ void store_result(int64_t sv, int64_t at, int my_idx, const SubVec<SUB> &s, const void *cb, int ct, bool aligned, void *idx,
                                             int it, const KeyXform &kx, int lane, bool live) {
    if (live) st_idx(idx, it, at, my_idx);
    if constexpr (LT > 0) {
        if (kx.k_tilde != nullptr && live) {
#pragma unroll
            for (int e = 0; e < SUB; e += 4)
                *reinterpret_cast<float4 *>(kx.k_tilde + sv * SUB + e) = make_float4(s.xf[e], s.xf[e + 1], s.xf[e + 2], s.xf[e + 3]);
        }
        if (kx.k_hat != nullptr) {   // block-uniform
            float row[SUB], c[8];
            load_centroid<SUB>(cb, ct, aligned, my_idx, row);
#pragma unroll
            for (int e = 0; e < 8; ++e) c[e] = e < SUB ? row[e] : 0.f;
            wht_lanes<SUB, LT>(c, lane);
#pragma unroll
            for (int e = 0; e < SUB; ++e) c[e] = c[e] * kx.h * s.sm[e];
            if (live) {
                if (kx.hat_dtype == VQ_F32) {
#pragma unroll
                    for (int e = 0; e < SUB; e += 4)
                        *reinterpret_cast<float4 *>((float *)kx.k_hat + sv * SUB + e) = make_float4(c[e], c[e + 1], c[e + 2], c[e + 3]);
                } else {
                    u32 w[4];
#pragma unroll
                    for (int e = 0; e < SUB; e += 2) {
                        if (kx.hat_dtype == VQ_F16) w[e / 2] = pack_h2(c[e], c[e + 1]);
                        else w[e / 2] = (u32)f32_to_bf16(c[e]) | ((u32)f32_to_bf16(c[e + 1]) << 16);
                    }
                    if constexpr (SUB == 8) *reinterpret_cast<uint4 *>((u16 *)kx.k_hat + sv * 8) = make_uint4(w[0], w[1], w[2], w[3]);
                    else *reinterpret_cast<uint2 *>((u16 *)kx.k_hat + sv * 4) = make_uint2(w[0], w[1]);
                }
            }
        }
    }
}

// What one assignment works on.
struct AssignJob {
    const void *x;
    int xt;
    int64_t N;        // sub-vectors
    const void *cb;
    int ct, nc;
    void *idx;
    int it;
    KeyXform kx;
    // where indices go: runs of row_len of them row_stride apart (an index store with room to grow); 0: one after the other
    int64_t row_len, row_stride;
};

// ---- IMAGE: dynamic LDS holds the operand tiles of the whole codebook ---------------------------

template <int SUB, int LT, int WAVES, bool FINE>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(4, 4)))
void vq_assign_image_kernel(AssignJob j) {
    extern __shared__ __align__(16) u32 s_img[];
    __shared__ float s_red[WAVES];
    constexpr int IW = image_words<SUB>();
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntiles = (j.nc + 63) / 64 * 2;   // an even number
    const bool aligned = (reinterpret_cast<uintptr_t>(j.cb) & 15u) == 0;

    float cmax2 = 0.f, kept[FINE ? SUB : 1];
    static_assert(!FINE || kFineC <= 64 * WAVES, "a thread reads one row");
    if constexpr (FINE) {   // one row a thread, read once: of a small call the second read's wait shows
        load_centroid<SUB>(j.cb, j.ct, aligned, min(tid, j.nc - 1), kept);
        cmax2 = norm2<SUB>(kept);
        cmax2 = cmax2 == cmax2 ? cmax2 : 0.f;
    } else {
        for (int c = tid; c < j.nc; c += 64 * WAVES) {
            float row[SUB];
            load_centroid<SUB>(j.cb, j.ct, aligned, c, row);
            cmax2 = fmaxf(cmax2, norm2<SUB>(row));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cmax2 = fmaxf(cmax2, __shfl_xor(cmax2, o));
    if (lane == 0) s_red[wave] = cmax2;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) cmax2 = fmaxf(cmax2, s_red[w]);
    const float cs = codebook_scale(cmax2);
    auto put = [&](int c, const u32 *img) {
#pragma unroll
        for (int e = 0; e < IW; e += 2) *reinterpret_cast<uint2 *>(&s_img[c * IW + e]) = make_uint2(img[e], img[e + 1]);
    };
    u32 img[IW];
    if constexpr (FINE) {
        if (tid < ntiles * 32) {
            if (tid < j.nc) centroid_image<SUB>(kept, cs, img);
            else pad_image<SUB>(img);
            put(tid, img);
        }
    } else {
        for (int c = tid; c < j.nc; c += 64 * WAVES) {
            float row[SUB];
            load_centroid<SUB>(j.cb, j.ct, aligned, c, row);
            centroid_image<SUB>(row, cs, img);
            put(c, img);
        }
        pad_image<SUB>(img);
        for (int c = j.nc + tid; c < ntiles * 32; c += 64 * WAVES) put(c, img);
    }
    __syncthreads();

    const u32 *a_ptr = s_img + (lane & 31) * IW + half * (SUB == 4 ? 2 : 4);
    const u32 mask = ~127u;
    // steps go to the blocks first, then to a block's waves: fewer steps than waves leave every CU its share
    const int64_t n_steps = (j.N + 63) / 64, stride = (int64_t)gridDim.x * WAVES;
    int64_t step = (int64_t)wave * gridDim.x + blockIdx.x;
    uint4 raw = load_raw<SUB>(j.x, j.xt, step * 64 + lane, step * 64 + lane < j.N);
    for (; step < n_steps; step += stride) {
        const int64_t sv = step * 64 + lane;
        const bool live = sv < j.N;
        SubVec<SUB> s;
        take_subvec<SUB, LT>(s, j.x, j.xt, raw, sv, live, lane, j.kx);
        {
            const int64_t nx = sv + stride * 64;
            raw = load_raw<SUB>(j.x, j.xt, nx, nx < j.N);
        }
        make_operands<SUB>(s, cs);
        u32 k1[2] = {~0u, ~0u}, k2[2] = {~0u, ~0u};
        auto product = [&](const u32 *ap, f32x16 *D) {
            const f32x16 zero = {};
            if constexpr (SUB == 4) {
                const uint2 p = *reinterpret_cast<const uint2 *>(ap), q = *reinterpret_cast<const uint2 *>(ap + 2);
                const f16x8 A = h8(p.x, p.y, q.x, q.y);
#pragma unroll
                for (int b = 0; b < 2; ++b) D[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, s.B1[b], zero, 0, 0, 0);
            } else {
                // words 0..3 / 4..7 of the first product, 0..3 / 8..11 of the second
                const f16x8 A1 = *reinterpret_cast<const f16x8 *>(ap), A2 = *reinterpret_cast<const f16x8 *>(ap + half * 4);
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    D[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A1, s.B1[b], zero, 0, 0, 0);
                    D[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A2, s.B2[b], D[b], 0, 0, 0);
                }
            }
        };
        const u32 *ap = a_ptr;
        auto track = [&](int b, const f32x16 &d, int t) {
            if constexpr (FINE) keep_quarters(k1[b], k2[b], d, mask, t);
            else keep_two(k1[b], k2[b], cell_key(d, mask, t));
        };
        f32x16 D[2];
        if constexpr (SUB == 4) {   // one tile's products are on their way while the other's scores are reduced
            f32x16 E[2];
            product(ap, D);
#pragma unroll 1
            for (int t = 0; t < ntiles; t += 2) {
                ap += 32 * IW;
                product(ap, E);
#pragma unroll
                for (int b = 0; b < 2; ++b) track(b, D[b], t);
                if (t + 2 < ntiles) {
                    ap += 32 * IW;
                    product(ap, D);
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) track(b, E[b], t + 1);
            }
        } else {
#pragma unroll 1
            for (int t = 0; t < ntiles; ++t, ap += 32 * IW) {
                product(ap, D);
#pragma unroll
                for (int b = 0; b < 2; ++b) track(b, D[b], t);
            }
        }
        // both halves' cells of the lane's own sub-vector: column block = lane / 32
        swap_halves(k1[0], k1[1]);
        swap_halves(k2[0], k2[1]);
        const bool low_first = k1[0] <= k1[1];   // [0]: rows of lanes 0..31, [1]: of lanes 32..63
        const u32 f1 = low_first ? k1[0] : k1[1], o1 = low_first ? k1[1] : k1[0];
        const u32 n1 = low_first ? k2[0] : k2[1], n2 = low_first ? k2[1] : k2[0];
        const int h1 = low_first ? 0 : 1;
        const float lim = __uint_as_float(f1) + margin<SUB>(s, f1);
        const bool second = !(__uint_as_float(o1) > lim);             // a cell of the other half may hold the winner
        const bool all = s.far || !(__uint_as_float(n1) > lim) || (second && !(__uint_as_float(n2) > lim));
        float dbest = INFINITY;
        int my_idx = 0;
        auto eval_cell = [&](u32 key, int hf) {
            constexpr int ALL = FINE ? 4 : 16, N = FINE || SUB == 8 ? 4 : 8;   // rows, and rows in flight: more would spill
#pragma unroll
            for (int g = 0; g < ALL; g += N) {
                int c[N];
                float row[N][SUB];
#pragma unroll
                for (int r = 0; r < N; ++r) {
                    const int first = FINE ? cell_centroid((key & 127u) >> 2, hf, key & 3u) : cell_centroid(key, hf, (g + r) >> 2);
                    c[r] = min(first + (r & 3), j.nc - 1);
                }
                load_centroids<SUB, N>(j.cb, j.ct, aligned, c, row);
#pragma unroll
                for (int r = 0; r < N; ++r) take_nearer(dbest, my_idx, exact_dist<SUB>(s.xf, row[r]), c[r]);
            }
        };
        my_idx = 0x7fffffff;
        eval_cell(f1, h1);
        if (__any(second)) { if (second) eval_cell(o1, 1 - h1); }
        const unsigned long long m = __ballot(all);
        if (m != 0) scan_all<SUB>(m, s.xf, j.cb, j.ct, aligned, j.nc, lane, my_idx);
        store_result<SUB, LT>(sv, sv, my_idx, s, j.cb, j.ct, aligned, j.idx, j.it, j.kx, lane, live);
    }
}

// The partner of a reduction over 16 lanes at step O = 1, 2, 4, 8, without a trip through LDS: 4 and 8 mirror the lanes of eight and
// sixteen, which after the steps before them hold the same in fours and eights.
template <int O, typename V> __device__ __forceinline__ V near_lane(V x) {
    static_assert(sizeof(V) == 4 && (O == 1 || O == 2 || O == 4 || O == 8), "a word, one of four steps");
    constexpr int CTRL = O == 1 ? 0xB1 : O == 2 ? 0x4E : O == 4 ? 0x141 : 0x140;
    const int i = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xF, 0xF, false));
}
template <class F> __device__ __forceinline__ void over_16_lanes(const F &step) {
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 4>{});
    step(std::integral_constant<int, 8>{});
}

// ---- SPLIT: one block for 64 sub-vectors, the tiles shared out over its waves -------------------

template <int WAVES> struct SplitLds {
    float red[WAVES];
    u32 keys[64][WAVES][4];   // of a sub-vector, wave by wave: two smallest cells of each half
    float xf[64][8];
    float x2[64];
    int idx[64];
};

// TW: tiles a wave takes at most
template <int SUB, int LT, int WAVES, int TW>
__device__ __forceinline__ void assign_split(const AssignJob &j, int64_t block, SplitLds<WAVES> &lds) {
    constexpr int IW = image_words<SUB>();
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntiles = (j.nc + 31) / 32;
    const bool aligned = (reinterpret_cast<uintptr_t>(j.cb) & 15u) == 0;
    const int64_t sv = block * 64 + lane;
    const bool live = sv < j.N;
    const uint4 raw = load_raw<SUB>(j.x, j.xt, sv, live);
    int rc[TW];
    float row[TW][SUB];
    float cmax2 = 0.f;
#pragma unroll
    for (int i = 0; i < TW; ++i) rc[i] = min((wave + i * WAVES) * 32 + (lane & 31), j.nc - 1);   // tiles wave, wave + WAVES, ..; past the end: the last centroid again (in its own tile, whose two cells are both looked at)
    load_centroids<SUB, TW>(j.cb, j.ct, aligned, rc, row);
#pragma unroll
    for (int i = 0; i < TW; ++i) cmax2 = fmaxf(cmax2, norm2<SUB>(row[i]));
    over_16_lanes([&](auto o) { cmax2 = fmaxf(cmax2, near_lane<o()>(cmax2)); });
    cmax2 = fmaxf(cmax2, __shfl_xor(cmax2, 16));
    if (lane == 0) lds.red[wave] = cmax2;
    SubVec<SUB> s;
    take_subvec<SUB, LT>(s, j.x, j.xt, raw, sv, live, lane, j.kx);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) cmax2 = fmaxf(cmax2, lds.red[w]);
    const float cs = codebook_scale(cmax2);
    make_operands<SUB>(s, cs);
    if (wave == 0) {
#pragma unroll
        for (int e = 0; e < SUB; e += 4) *reinterpret_cast<float4 *>(&lds.xf[lane][e]) = make_float4(s.xf[e], s.xf[e + 1], s.xf[e + 2], s.xf[e + 3]);
        lds.x2[lane] = s.far ? -1.f : s.x2;
    }
    u32 k1[2] = {~0u, ~0u}, k2[2] = {~0u, ~0u};
    const u32 mask = ~127u;
#pragma unroll
    for (int i = 0; i < TW; ++i) {
        const int t = wave + i * WAVES;
        if (t < ntiles) {   // wave-uniform
            u32 img[IW];
            centroid_image<SUB>(row[i], cs, img);
            f32x16 D[2];
            const f32x16 zero = {};
            if constexpr (SUB == 4) {
                const f16x8 A = h8(half ? img[2] : img[0], half ? img[3] : img[1], half ? img[4] : img[2], half ? img[5] : img[3]);
#pragma unroll
                for (int b = 0; b < 2; ++b) D[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, s.B1[b], zero, 0, 0, 0);
            } else {
                const f16x8 A1 = h8(half ? img[4] : img[0], half ? img[5] : img[1], half ? img[6] : img[2], half ? img[7] : img[3]);
                const f16x8 A2 = h8(half ? img[8] : img[0], half ? img[9] : img[1], half ? 0u : img[2], half ? 0u : img[3]);
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    D[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A1, s.B1[b], zero, 0, 0, 0);
                    D[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A2, s.B2[b], D[b], 0, 0, 0);
                }
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) keep_two(k1[b], k2[b], cell_key(D[b], mask, t));
        }
    }
    swap_halves(k1[0], k1[1]);
    swap_halves(k2[0], k2[1]);
    *reinterpret_cast<uint4 *>(&lds.keys[lane][wave][0]) = make_uint4(k1[0], k2[0], k1[1], k2[1]);
    __syncthreads();

    // merge: WAVES lanes a sub-vector, each with one wave's four cells
    const int g = tid / WAVES, l = tid % WAVES;   // sub-vector of the block, lane of its group
    {
        const uint4 e = *reinterpret_cast<const uint4 *>(&lds.keys[g][l][0]);
        // a tracker is (wave, half); of its two cells the first can lead, the second bounds what it dropped
        u32 f1 = min(e.x, e.z), f2 = max(e.x, e.z), bound = min(e.y, e.w);
        int o1 = 2 * l + (e.z < e.x), o2 = 2 * l + !(e.z < e.x);
        static_assert(WAVES == 16, "the lanes of a sub-vector");
        over_16_lanes([&](auto o) {
            const u32 g1 = near_lane<o()>(f1), g2 = near_lane<o()>(f2);
            const int p1 = near_lane<o()>(o1), p2 = near_lane<o()>(o2);
            bound = min(bound, near_lane<o()>(bound));
            const bool mine = f1 < g1 || (f1 == g1 && o1 < p1);
            // the second of the pair, and what falls out joins the bound
            const u32 a = mine ? f2 : g2, b = mine ? g1 : f1, c = mine ? g2 : f2;
            const int pa = mine ? o2 : p2, pb = mine ? p1 : o1;
            f1 = mine ? f1 : g1;
            o1 = mine ? o1 : p1;
            const bool keep = a < b || (a == b && pa < pb);
            f2 = keep ? a : b;
            o2 = keep ? pa : pb;
            bound = min(bound, min(keep ? b : a, c));
        });
        SubVec<SUB> v;
        v.x2 = lds.x2[g];
        const bool far = v.x2 < 0.f;
        float xs[SUB];
#pragma unroll
        for (int e = 0; e < SUB; e += 4) {
            const float4 t = *reinterpret_cast<const float4 *>(&lds.xf[g][e]);
            xs[e] = t.x; xs[e + 1] = t.y; xs[e + 2] = t.z; xs[e + 3] = t.w;
        }
        const float lim = __uint_as_float(f1) + margin<SUB>(v, f1);
        // (a codebook of one tile is its two cells: nothing was dropped that a bound stands for)
        const bool second = !(__uint_as_float(f2) > lim), all = far || (ntiles > 1 && !(__uint_as_float(bound) > lim));
        float d = INFINITY;
        int i = 0x7fffffff;
        // sixteen rows of a cell, 16 / WAVES a lane
#pragma unroll
        for (int k = 0; k < 16 / WAVES; ++k) {
            const int r = l * (16 / WAVES) + k, c = min(cell_centroid(f1, o1 & 1, r >> 2) + (r & 3), j.nc - 1);
            float rw[SUB];
            load_centroid<SUB>(j.cb, j.ct, aligned, c, rw);
            take_nearer(d, i, exact_dist<SUB>(xs, rw), c);
        }
        if (__any(second)) {
            if (second) {
#pragma unroll
                for (int k = 0; k < 16 / WAVES; ++k) {
                    const int r = l * (16 / WAVES) + k, c = min(cell_centroid(f2, o2 & 1, r >> 2) + (r & 3), j.nc - 1);
                    float rw[SUB];
                    load_centroid<SUB>(j.cb, j.ct, aligned, c, rw);
                    take_nearer(d, i, exact_dist<SUB>(xs, rw), c);
                }
            }
        }
        over_16_lanes([&](auto o) { take_nearer(d, i, near_lane<o()>(d), near_lane<o()>(i)); });
        // one lane of each group (a cell without a distance below infinity decides nothing)
        const unsigned long long m = __ballot((all || !(d < INFINITY)) && l == 0);
        if (m != 0) scan_all<SUB>(m, xs, j.cb, j.ct, aligned, j.nc, lane, i);
        if (l == 0) lds.idx[g] = i;
    }
    __syncthreads();
    const int64_t at = j.row_len == 0 ? sv : (int64_t)((u32)sv / (u32)j.row_len) * j.row_stride + (u32)sv % (u32)j.row_len;
    if (wave == 0) store_result<SUB, LT>(sv, at, lds.idx[lane], s, j.cb, j.ct, aligned, j.idx, j.it, j.kx, lane, live);
}

template <int SUB, int LT, int WAVES, int TW>
__global__ __launch_bounds__(64 * WAVES) void vq_assign_split_kernel(AssignJob j) {
    __shared__ SplitLds<WAVES> lds;
    assign_split<SUB, LT, WAVES, TW>(j, blockIdx.x, lds);
}

// A decode step's keys and values, SPLIT both, in one launch that writes into the index store: the first key_blocks blocks take the
// keys, the others the values beside them.  What bounds a few tokens is one block's latency, then launches and the
// host: apart it was a launch each and two strided copies (2 tokens, 8 heads of 128, 4096 x 4 and 256 x 8 centroids:
// 10.8 + 5.0 + 2 + 1.9 us and their gaps, now 10.8; 11.4 with the reductions over a sub-vector's lanes as LDS permutes).  Codebooks of every size take it, though alone SPLIT is the form for more
// than kSplitC centroids: 1 to 32 tokens, apart with the copies / here, in one graph, 256 x 8 keys and values 13.8-16.9 / 8.9-9.2
// us, 1024 x 8 keys 20-24 / 9.3-9.8, 32 x 8 keys and values 11.7-14.9 / 8.7-9.0.
template <int SUB, int LT>
__global__ __launch_bounds__(1024) void vq_encode_step_kernel(AssignJob jk, AssignJob jv, int key_blocks, int v_sub) {
    __shared__ SplitLds<16> lds;
    if ((int)blockIdx.x < key_blocks) assign_split<SUB, LT, 16, (SUB == 8 ? 4 : 8)>(jk, blockIdx.x, lds);
    else if (v_sub == 8) assign_split<8, 0, 16, 4>(jv, (int)blockIdx.x - key_blocks, lds);
    else assign_split<4, 0, 16, 8>(jv, (int)blockIdx.x - key_blocks, lds);
}

// ---- launch -----------------------------------------------------------------------------------

template <int SUB, int LT, int WAVES, bool FINE>
static void launch_image(const AssignJob &j, size_t image, int blocks_per_cu, hipStream_t st) {
    auto kernel = vq_assign_image_kernel<SUB, LT, WAVES, FINE>;
    // more than 64 KB of block-shared memory has to be allowed per kernel and device, once (a second
    // thread that gets here first repeats the same call)
    static std::atomic<bool> allowed[64] = {};
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev < 0 || dev >= 64 || !allowed[dev].load(std::memory_order_acquire)) {
        (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 256);
        if (dev >= 0 && dev < 64) allowed[dev].store(true, std::memory_order_release);
    }
    int64_t blocks = cdiv(j.N, 64);
    if (blocks > 256 * blocks_per_cu) blocks = 256 * blocks_per_cu;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(64 * WAVES), image, st, j);
}

template <int SUB, int LT> static bool launch_job(const AssignJob &j, hipStream_t st) {
    if (j.nc > (SUB == 8 ? VM_MAXC / 2 : VM_MAXC)) return false;
    const size_t image = (size_t)((j.nc + 63) / 64) * 64 * image_words<SUB>() * 4;
    if (j.nc <= kFineC) launch_image<SUB, LT, 8, true>(j, image, 2, st);
    else if (j.nc > kSplitC && j.N <= kSplitMax)
        hipLaunchKernelGGL((vq_assign_split_kernel<SUB, LT, 16, (SUB == 8 ? 4 : 8)>), dim3((unsigned)cdiv(j.N, 64)), dim3(1024), 0, st, j);
    else if (image <= 78 * 1024) launch_image<SUB, LT, 8, false>(j, image, 2, st);
    else launch_image<SUB, LT, 16, false>(j, image, 1, st);
    return true;
}

bool launch_assign_mfma(const void *x, int xt, int64_t N, const void *cb, int ct, int nc, int sub, void *idx, int it,
                        hipStream_t st) {
    if (!(sub == 4 || sub == 8)) return false;
    if (xt != VQ_F32 && ((uintptr_t)x & (sub == 8 ? 15u : 7u))) return false;
    const AssignJob j = {x, xt, N, cb, ct, nc, idx, it, {}, 0, 0};
    return sub == 8 ? launch_job<8, 0>(j, st) : launch_job<4, 0>(j, st);
}

bool launch_encode_keys_mfma(const void *keys, int kt, int64_t B, int64_t heads, int64_t S, int64_t D, const float *smooth,
                             int smooth_rows, float h, const void *cb, int ct, int nc, int sub, void *idx, int it, void *k_hat,
                             float *k_tilde, hipStream_t st) {
    if (!(sub == 4 || sub == 8) || D % sub != 0 || B * heads * S > 0x7fffffff) return false;
    const int64_t lt = D / sub;
    if (!(lt == 8 || lt == 16 || lt == 32 || lt == 64)) return false;
    if (((uintptr_t)keys | (uintptr_t)k_hat | (uintptr_t)k_tilde | (uintptr_t)smooth) & 15u) return false;
    const AssignJob j = {keys, kt, B * heads * S * lt, cb, ct, nc, idx, it, {smooth, smooth_rows, heads, S, h, k_hat, kt, k_tilde}, 0, 0};
#define VQ_ENC(SUB, LT) return launch_job<SUB, LT>(j, st)
    if (sub == 8) { if (lt == 8) VQ_ENC(8, 8); else if (lt == 16) VQ_ENC(8, 16); else if (lt == 32) VQ_ENC(8, 32); else VQ_ENC(8, 64); }
    else { if (lt == 8) VQ_ENC(4, 8); else if (lt == 16) VQ_ENC(4, 16); else if (lt == 32) VQ_ENC(4, 32); else VQ_ENC(4, 64); }
#undef VQ_ENC
}

bool launch_encode_step_mfma(const EncodeSide &k, const EncodeSide &v, int64_t B, int64_t heads, int64_t S, int64_t D, const float *smooth,
                             int smooth_rows, float h, int64_t cap, hipStream_t st) {
    const int64_t rows = B * heads;
    for (const EncodeSide *e : {&k, &v}) {
        if (!(e->sub == 4 || e->sub == 8) || D % e->sub != 0 || e->nc > (e->sub == 8 ? VM_MAXC / 2 : VM_MAXC)) return false;
        if (((uintptr_t)e->x & 15u) != 0) return false;
    }
    const int64_t lt = D / k.sub, lv = D / v.sub;
    if (!(lt == 8 || lt == 16 || lt == 32 || lt == 64) || ((uintptr_t)smooth & 15u) != 0) return false;
    // one block a CU in all (1024 threads each): up to there the two sides run beside each other; beyond, the launches of
    // their own choose between the forms
    const int64_t kb = cdiv(rows * S * lt, 64), vb = cdiv(rows * S * lv, 64);
    if (kb + vb > 256) return false;
    const AssignJob jk = {k.x, k.xt, rows * S * lt, k.cb, k.ct, k.nc, k.idx, k.it, {smooth, smooth_rows, heads, S, h, nullptr, k.xt, nullptr},
                          S * lt, cap * lt};
    const AssignJob jv = {v.x, v.xt, rows * S * lv, v.cb, v.ct, v.nc, v.idx, v.it, {}, S * lv, cap * lv};
#define VQ_STEP(SUB, LT)                                                                                                      \
    hipLaunchKernelGGL((vq_encode_step_kernel<SUB, LT>), dim3((unsigned)(kb + vb)), dim3(1024), 0, st, jk, jv, (int)kb, v.sub)
    if (k.sub == 8) { if (lt == 8) VQ_STEP(8, 8); else if (lt == 16) VQ_STEP(8, 16); else if (lt == 32) VQ_STEP(8, 32); else VQ_STEP(8, 64); }
    else { if (lt == 8) VQ_STEP(4, 8); else if (lt == 16) VQ_STEP(4, 16); else if (lt == 32) VQ_STEP(4, 32); else VQ_STEP(4, 64); }
#undef VQ_STEP
    return true;
}

}  // namespace vq
