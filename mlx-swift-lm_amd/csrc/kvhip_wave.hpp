// Wavefront reductions and the base-two exponential of the split-sequence decode kernels and their merge.
#pragma once
#include <hip/hip_runtime.h>

namespace kvhip {

constexpr float LOG2E = 1.4426950408889634f;

// v_exp_f32 without the denormal-range fix-up (results below 2^-126 flush to zero)
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Wavefront reductions on the data-parallel-primitive path (no LDS round trips): two quad
// permutes and two row mirrors leave each row of 16 lanes reduced, two row broadcasts
// carry the rows into lane 63, which is read out as a wave-uniform scalar.
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_take(float v) {  // v of the lane CTRL names; own v outside ROWS
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v),
                                                                 CTRL, ROWS, 0xF, false));
}
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_take<0xB1, 0xF>(v));   // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_take<0x4E, 0xF>(v));   // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_take<0x141, 0xF>(v));  // row_half_mirror
    v = fmaxf(v, dpp_take<0x140, 0xF>(v));  // row_mirror
    v = fmaxf(v, dpp_take<0x142, 0xA>(v));  // row_bcast15 into rows 1 and 3
    v = fmaxf(v, dpp_take<0x143, 0xC>(v));  // row_bcast31 into rows 2 and 3
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_take<0xB1, 0xF>(v);
    v += dpp_take<0x4E, 0xF>(v);
    v += dpp_take<0x141, 0xF>(v);
    v += dpp_take<0x140, 0xF>(v);
    // the broadcast steps must add only into the rows they target
    const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false));
    v += r1;
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xC, 0xF, false));
    v += r2;
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// inclusive prefix sums over the lanes
__device__ __forceinline__ float wave_scan(float v) {
#define KV_SCAN_STEP(CTRL, ROWS) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROWS, 0xF, true))
    KV_SCAN_STEP(0x111, 0xF);  // row_shr:1, 2, 4, 8
    KV_SCAN_STEP(0x112, 0xF);
    KV_SCAN_STEP(0x114, 0xF);
    KV_SCAN_STEP(0x118, 0xF);
#undef KV_SCAN_STEP
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false));  // row_bcast15 into rows 1 and 3
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xC, 0xF, false));  // row_bcast31 into rows 2 and 3
    return v;
}

}  // namespace kvhip
