// Wavefront reductions and the base-two exponential of the split-sequence decode kernels and their merge.
#pragma once
#include <hip/hip_runtime.h>

namespace kvhip {

constexpr float LOG2E = 1.4426950408889634f;

// v_exp_f32 without the denormal-range fix-up (results below 2^-126 flush to zero)
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Wavefront reductions on the data-parallel-primitive path (no LDS round trips): two quad
// permutes and two row mirrors leave each row of 16 lanes reduced, two row broadcasts
// carry the rows into lane 63, which is read out as a wave-uniform scalar.  Written as assembly, an instruction a step:
// through the permuting-move builtin a step is a copy, a wait, the move and the sum or (quieting) maximum.  A step waits two
// instructions for the one before it: N values are reduced in turn, one value waits.
#define KV_DPP_STEP(OP, V, CTRL) #OP "_dpp " V ", " V ", " V " " CTRL "\n\t"
#define KV_DPP_1(OP, CTRL) KV_DPP_STEP(OP, "%0", CTRL) "s_nop 1\n\t"
#define KV_DPP_4(OP, CTRL) KV_DPP_STEP(OP, "%0", CTRL) KV_DPP_STEP(OP, "%1", CTRL) KV_DPP_STEP(OP, "%2", CTRL) KV_DPP_STEP(OP, "%3", CTRL)
#define KV_DPP_REDUCE(STEP, OP)                                                                            \
    "s_nop 1\n\t" STEP(OP, "quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf")                              \
    STEP(OP, "quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf") STEP(OP, "row_half_mirror row_mask:0xf bank_mask:0xf") \
    STEP(OP, "row_mirror row_mask:0xf bank_mask:0xf") STEP(OP, "row_bcast:15 row_mask:0xa bank_mask:0xf")   \
    STEP(OP, "row_bcast:31 row_mask:0xc bank_mask:0xf") "s_nop 1"
__device__ __forceinline__ float lane_63(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63)); }
__device__ __forceinline__ float wave_max(float v) {
    asm(KV_DPP_REDUCE(KV_DPP_1, v_max_f32) : "+v"(v));
    return lane_63(v);
}
__device__ __forceinline__ float wave_sum(float v) {
    asm(KV_DPP_REDUCE(KV_DPP_1, v_add_f32) : "+v"(v));
    return lane_63(v);
}
__device__ __forceinline__ void wave_max4(float (&v)[4]) {
    asm(KV_DPP_REDUCE(KV_DPP_4, v_max_f32) : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = lane_63(v[i]);
}
__device__ __forceinline__ void wave_sum4(float (&v)[4]) {
    asm(KV_DPP_REDUCE(KV_DPP_4, v_add_f32) : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = lane_63(v[i]);
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
