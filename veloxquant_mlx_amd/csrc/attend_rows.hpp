// Helpers of the vector-unit attention kernels (attend_rows.hip, attend_wide.hip).
#pragma once
#include "attend.hpp"
#include "attend_mfma.hpp"

namespace vq {

namespace {

constexpr int AR_NR = 4;   // query rows per block

__device__ __forceinline__ float ar_ld(const void *p, int tag, int64_t i) {
    if (tag == VQ_F16) return (float)((const f16 *)p)[i];
    if (tag == VQ_BF16) return bf16_to_f32(((const u16 *)p)[i]);
    return ((const float *)p)[i];
}
template <int CTRL> __device__ __forceinline__ float ar_dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
// sum over the aligned group of `lpt` lanes (4, 8, 16, 32 or 64), left in every lane of the group
__device__ __forceinline__ float ar_slot_sum(float x, int lpt) {
    x += ar_dpp<0xB1>(x);                    // quad_perm [1,0,3,2]
    x += ar_dpp<0x4E>(x);                    // quad_perm [2,3,0,1]
    if (lpt >= 8) x += ar_dpp<0x141>(x);     // row_half_mirror
    if (lpt >= 16) x += ar_dpp<0x140>(x);    // row_mirror
    if (lpt >= 32) x += __shfl_xor(x, 16);
    if (lpt >= 64) x += __shfl_xor(x, 32);
    return x;
}

}  // namespace

}  // namespace vq
