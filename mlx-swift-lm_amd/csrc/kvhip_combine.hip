// Merge of the partials that launches over several spans of the keys leave: [bh][span][row][D + 2] floats, an output row
// not yet normalised, its maximum and its sum.
#include "kvhip_device.hpp"
#include "kvhip_wave.hpp"

namespace kvhip {

namespace {

// Partials of the float32 and the head-size-512 kernels: weights by the library's exponential, which takes the difference
// without rounding it to base two first and has no smallest weight above 2^-149 (an infinite value reaches the output from
// a span whose weight is denormal, as it does within a span), and sums by fused multiply-adds.
template <int D, int DT> constexpr bool exact_merge() { return DT == 2 || D == 512; }
// the weight of a partial with maximum m beside the row's maximum mx
template <bool EXACT> __device__ __forceinline__ float part_weight(float m, float mx) {
    if (m == -INFINITY) return 0.f;
    return EXACT ? expf(m - mx) : fast_exp2((m - mx) * LOG2E);
}
template <bool EXACT> __device__ __forceinline__ float add_weighed(float sum, float w, float v) {
    return EXACT ? __builtin_fmaf(w, v, sum) : sum + w * v;
}
template <int DT> __device__ __forceinline__ void store_pair(void *out, size_t i, float o0, float o1) {
    if constexpr (DT == 2) *reinterpret_cast<kv_out2f *>(static_cast<float *>(out) + i) = kv_out2f{o0, o1};
    else *reinterpret_cast<kv_out2 *>(static_cast<uint16_t *>(out) + i) = DT == 0 ? pk_h2(o0, o1) : pk_bf2(o0, o1);
}

// grid (R, BH, D / CB), 256 threads: merge the span partials of CB columns of one query row and write them.
// A launch with few rows and many spans (a single sequence: 8 pairs, 32 to 512 spans each) lasts as long as its
// chain of memory round trips, so everything is asked for at once: a thread is (column pair, span group) and
// requests its first eight partial pairs before anything else, then the (max, sum) of up to two spans; the weights
// are formed while the columns are in flight, go through LDS, and the span groups' sums meet there at the end.  Wide rows
// are cut into blocks of columns so that one round of requests holds every span of the usual plans.
template <int D, int DT, int CB, bool SPANS>
__global__ void __launch_bounds__(256) combine_kernel(AttendArgs a, int nsplit, int rr, const int2 *spans) {
    static_assert(D % CB == 0, "whole blocks of columns");
    constexpr int CP = CB / 2;    // column pairs
    constexpr int NG = 256 / CP;  // span groups: 16 (32 columns), 8 (64), 6, 5, 4 (128)
    constexpr int UN = 8;         // loads in flight per thread and round
    constexpr bool EXACT = exact_merge<D, DT>();
    __shared__ float w_s[512];    // weight of each span for this row (nsplit <= 512)
    __shared__ float red_s[2][4];
    __shared__ kv_f2 acc_s[NG][CP];
    const int i = blockIdx.x, bh = blockIdx.y;
    const size_t sstride = (size_t)rr * (D + 2);
    size_t first_slot = (size_t)bh * nsplit;
    if constexpr (SPANS) {  // (a ragged batch's rows have spans in proportion to their keys: kvhip_mask.hpp)
        const int2 own = spans[bh];
        first_slot = own.x;
        nsplit = own.y;
    }
    // (rows of D + 2 floats, D even: every pair below is 8-byte aligned)
    const float *part = a.workspace + first_slot * sstride + (size_t)i * (D + 2);
    const int t = threadIdx.x, c0 = CB < D ? blockIdx.z * CB : 0;
    const int g = t / CP, cp = t - g * CP;
    const bool col = g < NG;
    auto pair_at = [&](int s, int c) { return *reinterpret_cast<const kv_f2 *>(part + (size_t)s * sstride + c); };
    kv_f2 v[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
        const int s = g + NG * u;
        v[u] = (col && s < nsplit) ? pair_at(s, c0 + 2 * cp) : kv_f2{0.f, 0.f};
    }
    kv_f2 ml[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) ml[u] = t + 256 * u < nsplit ? pair_at(t + 256 * u, D) : kv_f2{-INFINITY, 0.f};
    float mloc = wave_max(fmaxf(ml[0].x, ml[1].x));
    if ((t & 63) == 0) red_s[0][t >> 6] = mloc;
    __syncthreads();
    const float mx = fmaxf(fmaxf(red_s[0][0], red_s[0][1]), fmaxf(red_s[0][2], red_s[0][3]));
    float dloc = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const float w = part_weight<EXACT>(ml[u].x, mx);
        if (t + 256 * u < nsplit) w_s[t + 256 * u] = w;
        dloc += w * ml[u].y;
    }
    dloc = wave_sum(dloc);
    if ((t & 63) == 0) red_s[1][t >> 6] = dloc;
    __syncthreads();
    const float den = (red_s[1][0] + red_s[1][1]) + (red_s[1][2] + red_s[1][3]);
    kv_f2 num{0.f, 0.f};
#pragma unroll
    for (int u = 0; u < UN; ++u) {
        const int s = g + NG * u;
        if (col && s < nsplit) num = kv_f2{add_weighed<EXACT>(num.x, w_s[s], v[u].x), add_weighed<EXACT>(num.y, w_s[s], v[u].y)};
    }
    for (int s0 = g + NG * UN; col && s0 < nsplit; s0 += NG * UN) {  // more than 8 NG spans: further rounds
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int s = s0 + NG * u;
            v[u] = s < nsplit ? pair_at(s, c0 + 2 * cp) : kv_f2{0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int s = s0 + NG * u;
            if (s < nsplit) num = kv_f2{add_weighed<EXACT>(num.x, w_s[s], v[u].x), add_weighed<EXACT>(num.y, w_s[s], v[u].y)};
        }
    }
    if (col) acc_s[g][cp] = num;
    __syncthreads();
    if (t < CP) {
        kv_f2 o = acc_s[0][t];
#pragma unroll
        for (int k = 1; k < NG; ++k) o += acc_s[k][t];
        // (a pair's query rows lie one behind the other: Hq / Hkv heads of L rows)
        store_pair<DT>(a.out, ((size_t)bh * gridDim.x + i) * D + c0 + 2 * t, den > 0.f ? o.x / den : 0.f, den > 0.f ? o.y / den : 0.f);
    }
}

// The same merge for the prefill tiles' key-range parts: many query rows, at most 8 parts.  D / 4 lanes per query row,
// four adjacent columns each, as many rows per workgroup as fit 256 threads; no LDS and no barrier (the
// per-row workgroups above spend their time being launched: 22 us for 16 384 rows of 256 columns).  Bound by the latency of
// its loads: every part's columns, maximum and sum are requested before any of them is looked at (parts up to MAXP = 2, 4
// or 8; the numbers beyond nsplit repeat the last one's loads and are left out of the sums).  With the maxima read first and a part's columns
// behind a branch of their own it took 12.0 us where it takes 7.6 (16 384 rows of 128, 3 or 4 parts), 11.1 where 9.6 (256
// columns).
// Decode launches keep the kernel above: with few rows and many parts it has the loads of a column in flight together
// (a ring decode of 2 rows of 16 parts: 29.1 us per step against 31.7 us with this one).
template <int D, int DT, int MAXP>
__global__ void __launch_bounds__(256) combine_rows_kernel(AttendArgs a, int nsplit, int rr) {
    constexpr int LPR = D / 4, RPW = 256 / LPR;
    constexpr bool EXACT = exact_merge<D, DT>();
    const int in_wg = threadIdx.x / LPR, c = 4 * (threadIdx.x % LPR);
    const int i = blockIdx.x * RPW + in_wg, bh = blockIdx.y;
    if (in_wg >= RPW || i >= rr) return;
    const size_t sstride = (size_t)rr * (D + 2);
    const float *part = a.workspace + (size_t)bh * nsplit * sstride + (size_t)i * (D + 2);
    kv_f2 ml[MAXP], p[MAXP][2];  // (a row of partials is 8-byte aligned: D + 2 floats)
#pragma unroll
    for (int s = 0; s < MAXP; ++s) {
        const float *row = part + min(s, nsplit - 1) * sstride;
        ml[s] = *reinterpret_cast<const kv_f2 *>(row + D);
        p[s][0] = *reinterpret_cast<const kv_f2 *>(row + c);
        p[s][1] = *reinterpret_cast<const kv_f2 *>(row + c + 2);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int s = 0; s < MAXP; ++s) mx = fmaxf(mx, ml[s].x);
    float den = 0.f, num[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < MAXP; ++s) {
        const float w = part_weight<EXACT>(ml[s].x, mx);
        const bool own = s < nsplit;
        den = own ? add_weighed<EXACT>(den, w, ml[s].y) : den;
        num[0] = own ? add_weighed<EXACT>(num[0], w, p[s][0].x) : num[0];
        num[1] = own ? add_weighed<EXACT>(num[1], w, p[s][0].y) : num[1];
        num[2] = own ? add_weighed<EXACT>(num[2], w, p[s][1].x) : num[2];
        num[3] = own ? add_weighed<EXACT>(num[3], w, p[s][1].y) : num[3];
    }
    const size_t ooff = ((size_t)bh * rr + i) * D + c;  // (a pair's query rows lie one behind the other)
#pragma unroll
    for (int k = 0; k < 2; ++k) store_pair<DT>(a.out, ooff + 2 * k, den > 0.f ? num[2 * k] / den : 0.f, den > 0.f ? num[2 * k + 1] / den : 0.f);
}

template <int D, int DT, int CB> hipError_t merge(const AttendArgs &a, int nsplit, int rows, const int2 *spans, hipStream_t s) {
    const int R = (a.Hq / a.Hkv) * a.L;
    if (rows > 16 && nsplit <= 8 && rows == R) {  // the parts of prompt chunks
        constexpr int RPW = 256 / (D / 4);
        const dim3 grid((R + RPW - 1) / RPW, a.st.BH), block(256);
        if (nsplit <= 2) hipLaunchKernelGGL((combine_rows_kernel<D, DT, 2>), grid, block, 0, s, a, nsplit, rows);
        else if (nsplit <= 4) hipLaunchKernelGGL((combine_rows_kernel<D, DT, 4>), grid, block, 0, s, a, nsplit, rows);
        else hipLaunchKernelGGL((combine_rows_kernel<D, DT, 8>), grid, block, 0, s, a, nsplit, rows);
    } else {
        const dim3 grid(R, a.st.BH, D / CB), block(256);
        if constexpr (DT != 2 && D <= 256) {
            if (spans != nullptr) {
                hipLaunchKernelGGL((combine_kernel<D, DT, CB, true>), grid, block, 0, s, a, nsplit, rows, spans);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((combine_kernel<D, DT, CB, false>), grid, block, 0, s, a, nsplit, rows, spans);
    }
    return hipGetLastError();
}
template <int D, int CB> hipError_t merge_dtype(const AttendArgs &a, int nsplit, int rows, const int2 *spans, hipStream_t s) {
    if (a.st.dtype == KVHIP_F16) return merge<D, 0, CB>(a, nsplit, rows, spans, s);
    if (a.st.dtype == KVHIP_BF16) return merge<D, 1, CB>(a, nsplit, rows, spans, s);
    return merge<D, 2, CB>(a, nsplit, rows, spans, s);
}

}  // namespace

bool combine_supported(const Store &s) {
    return s.Dv == 64 || s.Dv == 80 || s.Dv == 96 || s.Dv == 128 || s.Dv == 256 || s.Dv == 512;
}

// (the partials hold output columns: the head size of the values)
hipError_t launch_combine(const AttendArgs &a, int nsplit, int rows, hipStream_t s, const int2 *spans) {
    if (a.st.Dv == 64) return merge_dtype<64, 64>(a, nsplit, rows, spans, s);
    if (a.st.Dv == 80) return merge_dtype<80, 80>(a, nsplit, rows, spans, s);
    if (a.st.Dv == 96) return merge_dtype<96, 96>(a, nsplit, rows, spans, s);
    // Blocks of fewer columns shorten a workgroup's chain, which is what a launch of few rows and many spans lasts, and are
    // workgroups more.  Whole steps, us, 64 / 128 columns at head size 128: 32 rows over 16 000 keys of 4 bits 9.2 / 10.4, 64 rows
    // 11.0 / 12.0, 128 rows over 2000 keys 7.3 / 7.5, 512 rows 10.6 / 10.8 (64q/8kv) and 13.3 / 13.1 (32q), 1024 rows 14.2 / 13.8, 2048
    // 19.2 / 17.6.  32 / 64 columns at 512, bfloat16: 8 rows over 4000 keys 8.3 / 9.2, 16 rows 11.4 / 11.9, 32 rows 12.4 / 12.9 and 12.6 /
    // 13.0, 64 rows 13.8 / 13.7, 128 rows 19.0 / 18.6 and 25.7 / 24.9.
    const size_t all = (size_t)(a.Hq / a.Hkv) * a.L * a.st.BH;
    if (a.st.Dv == 128) return all <= 512 ? merge_dtype<128, 64>(a, nsplit, rows, spans, s) : merge_dtype<128, 128>(a, nsplit, rows, spans, s);
    if (a.st.Dv == 256) return merge_dtype<256, 128>(a, nsplit, rows, spans, s);
    if (a.st.Dv == 512) return all <= 32 ? merge_dtype<512, 32>(a, nsplit, rows, spans, s) : merge_dtype<512, 64>(a, nsplit, rows, spans, s);
    return hipErrorInvalidValue;
}

}  // namespace kvhip
