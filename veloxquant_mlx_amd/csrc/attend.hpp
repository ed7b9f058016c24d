// Declarations shared by the attention translation units.
#pragma once
#include "common.hpp"

namespace vq {

// A call as the library runs it: the caller's argument block and what vq_attend_ext adds to it.  One length a sequence travels in
// the block's own fields -- packed_lens the int64 list, tail_lens null, a form that no caller's block has -- and the kernels
// that know nothing of pairs take the block alone: two more fields in every kernel's arguments made the sixteen launches of an 8k
// prefill 3 us longer in all.
struct AttendCall : vq_attend_args {
    int32_t pair_heads;   // > 0: kv heads of 64 channels, kept in pairs; the caller's kv head count (negative: not one)
    int32_t few_parts;    // 1: the plan with the fewest partials (scratch of a fixed size)
    AttendCall() = default;
    explicit AttendCall(const vq_attend_args &a, const vq_attend_ext *x = nullptr)
        : vq_attend_args(a), pair_heads(x == nullptr ? 0 : x->pair_heads == (int32_t)x->pair_heads ? (int32_t)x->pair_heads : -1), few_parts(0) {
        if (x != nullptr && x->seq_lens != nullptr) {
            packed_lens = reinterpret_cast<const int32_t *>(x->seq_lens);
            tail_lens = nullptr;
        }
    }
};

// live slots of every sequence, prefix and tail together (null: none, or two lists of lengths)
__device__ __host__ __forceinline__ const int64_t *seq_lens(const vq_attend_args &a) {
    return a.tail_lens == nullptr ? reinterpret_cast<const int64_t *>(a.packed_lens) : nullptr;
}

// a batch whose sequences differ in length: the block's copy of the arguments takes the lengths
// of its own sequence
__device__ __forceinline__ void take_sequence_lengths(vq_attend_args &a, int64_t b) {
    if (__builtin_expect(a.packed_lens == nullptr, 1)) return;
    if (const int64_t *lens = seq_lens(a)) {
        const int64_t n = lens[b], tail = n - a.n_packed;
        if (tail < a.n_tail) a.n_tail = tail < 0 ? 0 : tail;
        if (n < a.n_packed) a.n_packed = n;
    } else {
        a.n_packed = a.packed_lens[b];
        a.n_tail = a.tail_lens[b];
    }
}

// first slot a query at position `pos` (of Sq, aligned to the end of n_total slots) sees under a
// sliding window; 0 without one
__device__ __host__ __forceinline__ int64_t window_first(const vq_attend_args &a, int64_t n_total, int64_t pos) {
    const int64_t lo = n_total - a.Sq + pos + 1 - a.sliding_window;
    return a.sliding_window > 0 && lo > 0 ? lo : 0;
}

constexpr int EVEN_BLOCKS = 256;   // one to a CU

struct AttendPlan {
    int path;           // 0 generic waves, 1 MFMA decode (row tiles of <= 8), 2 MFMA prefill (LDS-staged, 64-row blocks),
                        // 3 vector-unit rows kernel (any head_dim / bit width, four query rows a block),
                        // 4 the same over byte codes, sixteen channels a lane (attend_wide.hip)
    int nsplit;         // splits along the tokens the main kernel covers
    int nparts;         // partials per query row handed to the merge kernel
    int64_t split_len;  // tokens per split (multiple of 64)
    // MFMA path: the block of split 0 also runs the fp16 tail and takes this many fewer
    // packed tokens (multiple of 64); split s covers packed tokens
    // [max(0, s*split_len - tail_equiv), min(n_packed, (s+1)*split_len - tail_equiv))
    int64_t tail_equiv;
    // MFMA path: a block works on the GQA group of one kv head at pq consecutive query
    // positions (eight heads of a group of more than eight, pq = 1); tiles such blocks per (batch, kv head)
    int pq, tiles;
    // MFMA decode path: deal token chunks to the waves round robin instead of on demand, so that
    // results are identical from run to run
    int fixed_order;
    // MFMA decode path, sequences of different lengths: a launch of EVEN_BLOCKS blocks that work split_len (at least the one above)
    // and the splits of every tile (at most nsplit) out from all lengths
    int even = 0;
    // rows kernel over the tail only: first partial it writes (-1: the whole context, partials 0 .. nsplit - 1)
    int part0 = -1;
};

// One output element from the split partials of its query row: p points at nparts records
// of `stride` floats (max in natural-log units, sum, accumulator[D]).  CH records are
// fetched at a time with independent loads (a round costs one memory latency, so callers with
// many records pick a large CH).
template <int CH>
__device__ __forceinline__ float merge_partials(const float *p, int nparts, int64_t stride, int64_t d) {
    float gm = -INFINITY, num = 0.f, den = 0.f;
    for (int s0 = 0; s0 < nparts; s0 += CH) {
        float m[CH], l[CH], o[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const float *q = p + (int64_t)(s0 + j < nparts ? s0 + j : s0) * stride;
            m[j] = q[0];
            l[j] = q[1];
            o[j] = q[2 + d];
        }
        // every load of the round is issued before the first use: left to itself the scheduler
        // weaves the maxima between the loads and waits for each record in turn
        __builtin_amdgcn_sched_barrier(0);
        float cm = gm;
#pragma unroll
        for (int j = 0; j < CH; ++j)
            if (s0 + j < nparts) cm = fmaxf(cm, m[j]);
        if (cm == -INFINITY) continue;   // nothing visible so far
        const float f0 = __expf(gm - cm);   // 0 on the first chunk
        num *= f0;
        den *= f0;
#pragma unroll
        for (int j = 0; j < CH; ++j)
            if (s0 + j < nparts && m[j] != -INFINITY) {
                const float f = __expf(m[j] - cm);
                den += l[j] * f;
                num += o[j] * f;
            }
        gm = cm;
    }
    return den > 0.f ? num / den : 0.f;
}
// The round size by the number of records: one round of loads when they fit.  The decode kernel that merges inside its launch
// (merge_rows) fetches whole records through LDS and adds them in rounds of the same sizes, in the same order;
// launch_merge_splits, of the vector kernels, has an order of its own.
constexpr int MERGE_FEW = 8, MERGE_SOME = 16, MERGE_MANY = 36;
__device__ __forceinline__ float merge_records(const float *p, int nparts, int64_t stride, int64_t d) {
    return nparts <= MERGE_FEW ? merge_partials<MERGE_FEW>(p, nparts, stride, d)
           : nparts <= MERGE_SOME ? merge_partials<MERGE_SOME>(p, nparts, stride, d)
                                  : merge_partials<MERGE_MANY>(p, nparts, stride, d);
}


// Decides kernel and split count from shapes, whether there are lengths and the order, so that the workspace query (`widest`: the order
// with the most partials) covers the launch.
AttendPlan plan_attend(const AttendCall &a, bool widest = false);

int launch_attend_generic(const AttendCall &a, int nsplit, int64_t split_len);
// vector-unit kernel with the kv head's bytes shared by its query heads (attend_rows.hip): whether it takes the
// shapes, its row tiling (positions per tile, tiles per (sequence, kv head)), the launch
bool rows_kernel_supported(const AttendCall &a);
void rows_tiling(const AttendCall &a, int &pq, int &tiles);
int launch_attend_rows(const AttendCall &a, const AttendPlan &p);
// the same kernel over the tail tokens only, in `runs` runs into partials `part0` on of `nparts` per query row
int launch_attend_rows_tail(const AttendCall &a, int part0, int runs, int nparts);
// byte codes, sixteen channels a lane (attend_wide.hip): whether it takes the shapes, its splits, the launch
bool wide_kernel_supported(const AttendCall &a);
void plan_attend_wide(const AttendCall &a, AttendPlan &p);
void launch_attend_wide(const AttendCall &a, const AttendPlan &p);
int launch_attend_merge(const AttendCall &a, int nparts);
// protected rows (AttendCall.sink_k): rewrites every output row from the partials in the
// workspace, with the stand-ins' weights taken out and the exact rows put in
void launch_sink_patch(const AttendCall &a, int nparts);
// merges partials [rows][nparts][D + 2] of (max, sum, accumulator) into out [rows][D]
void launch_merge_rows(const float *ws, int64_t rows, int nparts, int64_t D, void *out, int out_dtype, hipStream_t st);
// the same with a block a row where partials are many (sums in another order: not for launches whose other form merges
// inside the kernel)
void launch_merge_splits(const float *ws, int64_t rows, int nparts, int64_t D, void *out, int out_dtype, hipStream_t st);

// MFMA decode path (attend_mfma.hip)
bool mfma_decode_supported(const AttendCall &a);
int mfma_row_tiles(const AttendCall &a);
int mfma_positions_per_tile(const AttendCall &a);

// MFMA prefill path (attend_prefill.hip): packed prefix into partial slot 0, tail into slot 1
bool mfma_prefill_supported(const AttendCall &a);
int mfma_prefill_block_rows(const AttendCall &a);   // 64, or 256 when a kv head has that many query rows
// returns true when the kernel wrote the output itself (one run per row: nothing to merge)
bool launch_attend_mfma_prefill(const AttendCall &a, const AttendPlan &p);
// that case, from the shapes alone: such a launch writes no partials and needs no workspace
bool mfma_prefill_direct_output(const AttendCall &a, int nparts);
// whether a launch of the 256-row blocks takes its units from a.kv_tiles
bool mfma_prefill_uses_tiles(const AttendCall &a);
// writes tiles [first_unit, first_unit + n_units) of every (sequence, kv head); VQ_OK or an error code
int launch_prefill_tiles(const AttendCall &a, int64_t first_unit, int64_t n_units);
// returns true when the kernel also merged the partials (sync counters were given)
bool launch_attend_mfma_decode(const AttendCall &a, const AttendPlan &p);

}  // namespace vq
