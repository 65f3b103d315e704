// What a decode kernel's workgroup does with its wavefronts' partial results: joins them in LDS and writes output rows, or a
// partial of its span of the keys for the merge.
#pragma once
#include "kvhip_device.hpp"
#include "kvhip_wave.hpp"

namespace kvhip {

typedef float kv_f4 __attribute__((ext_vector_type(4)));

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
__device__ __forceinline__ kv_f4 normalised(kv_f4 v, float l) {
    if (!(l > 0.f)) return kv_f4{0.f, 0.f, 0.f, 0.f};
    const float r = 1.f / l;
    kv_f4 q;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float x = v[k] * r, y = __builtin_fmaf(__builtin_fmaf(-x, l, v[k]), r, x);
        q[k] = __builtin_isfinite(x) ? y : x;
    }
    return q;
}
// R rows, a thread to four columns of one: output rows row0 .. (`whole`), or partial `slot` of the workspace (RR rows of D
// columns, maximum, sum).
template <int D, int DT, int NW, int RR>
__device__ __forceinline__ void leave_rows(const AttendArgs &a, const WaveParts<D, NW, RR> &parts, int R, bool whole, size_t row0, size_t slot) {
    constexpr int LPR = D / 4, RPB = NW * 64 / LPR;
    const int c = 4 * (threadIdx.x % LPR);
    if (RPB * LPR < NW * 64 && threadIdx.x >= RPB * LPR) return;  // (96 columns: lanes left over)
#pragma unroll 1
    for (int i = threadIdx.x / LPR; i < R; i += RPB) {
        kv_f4 v{0.f, 0.f, 0.f, 0.f};
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            v += *reinterpret_cast<const kv_f4 *>(&parts.rows[w][i][c]);
            l += parts.l[w][i];
        }
        if (whole) {
            const kv_f4 o = normalised(v, l);
            *reinterpret_cast<kv_u2 *>(static_cast<uint16_t *>(a.out) + (row0 + i) * D + c) =
                DT == 0 ? kv_u2{pk_h2(o.x, o.y), pk_h2(o.z, o.w)} : kv_u2{pk_bf2(o.x, o.y), pk_bf2(o.z, o.w)};
        } else {
            float *part = a.workspace + (slot * RR + i) * (D + 2);
            *reinterpret_cast<kv_f2 *>(part + c) = kv_f2{v.x, v.y};
            *reinterpret_cast<kv_f2 *>(part + c + 2) = kv_f2{v.z, v.w};
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
