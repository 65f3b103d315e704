// What a decode kernel's workgroup does with its wavefronts' partial results: joins them in LDS and writes output rows, or a
// partial of its span of the keys for the merge.
#pragma once
#include "kvhip_device.hpp"
#include "kvhip_wave.hpp"

namespace kvhip {

// The wavefronts' maxima, and behind a barrier their rows and sums, weighed by exp2(own maximum - row's maximum) as they
// are written: what is left to do is to add them up.  (The weights formed by every thread that adds, an exponential per
// wavefront and column, cost the last wavefront 1100 cycles behind its last tile at four rows of 64; now 600.)
template <int D, int NW, int RR> struct WaveParts {
    float m[NW][RR], l[NW][RR];
    float rows[NW][RR][D + 4];  // (rows of one column block on different banks)
};
// the weight of a wavefront's part of row i, its maximum there being m
template <int D, int NW, int RR> __device__ __forceinline__ float wave_weight(const WaveParts<D, NW, RR> &parts, int i, float m) {
    float mx = parts.m[0][i];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, parts.m[w][i]);
    return m == -INFINITY ? 0.f : fast_exp2((m - mx) * LOG2E);
}
// v / l, a thread's columns by one division and a correction each
template <int N> __device__ __forceinline__ void normalise(float (&v)[N], float l) {
    const float r = 1.f / l;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const float x = v[k] * r, y = __builtin_fmaf(__builtin_fmaf(-x, l, v[k]), r, x);
        v[k] = !(l > 0.f) ? 0.f : __builtin_isfinite(x) ? y : x;
    }
}
// N adjacent elements of an output row
template <int DT, int N> __device__ __forceinline__ void store_columns(void *out, size_t i, const float (&v)[N]) {
    uint16_t *p = static_cast<uint16_t *>(out) + i;
    if constexpr (N == 1) {
        Elem<DT>::store(p, 0, v[0]);
    } else {
        uint32_t w[N / 2];
#pragma unroll
        for (int k = 0; k < N / 2; ++k) w[k] = DT == 0 ? pk_h2(v[2 * k], v[2 * k + 1]) : pk_bf2(v[2 * k], v[2 * k + 1]);
        if constexpr (N == 2) *reinterpret_cast<kv_out2 *>(p) = w[0];
        else *reinterpret_cast<kv_out4 *>(p) = kv_out4{w[0], w[1]};
    }
}
template <int N> __device__ __forceinline__ void store_floats(float *p, const float (&v)[N]) {  // (8-byte aligned where N > 1)
    if constexpr (N == 1) p[0] = v[0];
#pragma unroll
    for (int k = 0; k + 1 < N; k += 2) *reinterpret_cast<kv_f2 *>(p + k) = kv_f2{v[k], v[k + 1]};
}
// R rows, a thread to CPT columns of one (as few as leave no thread of a full workgroup without any): output rows row0 ..
// (`whole`), or partial `slot` of the workspace (RR rows of D columns, maximum, sum).
template <int D, int DT, int NW, int RR>
__device__ __forceinline__ void leave_rows(const AttendArgs &a, const WaveParts<D, NW, RR> &parts, int R, bool whole, size_t row0, size_t slot) {
    constexpr int EACH = RR * D / (NW * 64), CPT = EACH >= 4 ? 4 : EACH >= 2 ? 2 : 1;
    constexpr int LPR = D / CPT, RPB = NW * 64 / LPR;
    const int c = CPT * (threadIdx.x % LPR);
    if (RPB * LPR < NW * 64 && threadIdx.x >= RPB * LPR) return;  // (96 columns: lanes left over)
#pragma unroll 1
    for (int i = threadIdx.x / LPR; i < R; i += RPB) {
        float v[CPT], l = 0.f;
#pragma unroll
        for (int k = 0; k < CPT; ++k) v[k] = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
#pragma unroll
            for (int k = 0; k < CPT; ++k) v[k] += parts.rows[w][i][c + k];
            l += parts.l[w][i];
        }
        if (whole) {
            normalise(v, l);
            store_columns<DT>(a.out, (row0 + i) * D + c, v);
        } else {
            float *part = a.workspace + (slot * RR + i) * (D + 2);
            store_floats(part + c, v);
            if (c == 0) {
                float mx = parts.m[0][i];
#pragma unroll
                for (int w = 1; w < NW; ++w) mx = fmaxf(mx, parts.m[w][i]);
                *reinterpret_cast<kv_f2 *>(part + D) = kv_f2{mx, l};
            }
        }
    }
}

}  // namespace kvhip
