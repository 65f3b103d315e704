// Rotary position embedding as the append kernels and the query pass apply it: the angle and its sine and
// cosine, single elements (any shape), and 16-byte chunks (what the tuned kernels move).
#pragma once
#include "kvhip_device.hpp"

namespace kvhip {

// Sine and cosine of a remainder of at most pi/4 and the quadrant it was taken from.
__device__ __forceinline__ void rope_sincos_reduced(float x, int quad, float &sn, float &cs) {
    const float z = x * x;
    float s = __builtin_fmaf(z, 2.7557319223985893e-6f, -1.9841269841269841e-4f);
    s = __builtin_fmaf(z, s, 8.3333333333333332e-3f);
    s = __builtin_fmaf(z, s, -1.6666666666666667e-1f);
    s = __builtin_fmaf(x * z, s, x);
    float c = __builtin_fmaf(z, -2.7557319223985888e-7f, 2.4801587301587302e-5f);
    c = __builtin_fmaf(z, c, -1.3888888888888889e-3f);
    c = __builtin_fmaf(z, c, 4.1666666666666664e-2f);
    c = __builtin_fmaf(z, c, -0.5f);
    c = __builtin_fmaf(z, c, 1.0f);
    const float a = (quad & 1) ? c : s, b = (quad & 1) ? s : c;
    sn = (quad & 2) ? -a : a;
    cs = ((quad + 1) & 2) ? -b : b;
}

// The remainder and quadrant of an angle of 2^24 and more, by Payne and Hanek's method: the angle is m 2^e with an integer
// m < 2^24, and of 2/pi only the 64 bits from weight 2^(1 - e) on matter to the product modulo 4 (an error of the
// remainder below 2^-37).
__device__ __forceinline__ void rope_reduce_large(float theta, float &x, int &quad) {
    const uint32_t u = __float_as_uint(theta);
    const int at = (int)((u >> 23) & 255u) - 151;  // the first bit that matters: 0 .. 103 (104: infinite, NaN)
    const uint64_t m = (u & 0x7fffffu) | 0x800000u;
    constexpr uint64_t T0 = 0x517cc1b727220a94ull, T1 = 0xfe13abe8fa9a6ee0ull, T2 = 0x6db14acc9e21c820ull;  // 2/pi, the first bit has weight 1
    const uint64_t hi = at < 64 ? T0 : T1, lo = at < 64 ? T1 : T2;
    const uint64_t p = m * ((hi << (at & 63)) | ((lo >> 1) >> (63 - (at & 63))));  // times 2^62, modulo 4
    const uint64_t k = (p + (1ull << 61)) >> 62;
    x = at == 104 ? theta - theta : (float)((double)(int64_t)(p - (k << 62)) * 3.4061215800865545e-19);  // pi/2 2^-62
    quad = (int)k;
    if (u >> 31) {
        x = -x;
        quad = -quad;
    }
}
// A function of its own: positions times frequencies do not get there in ordinary use, and a copy of it beside each of the
// sixteen short ones of a chunk kept the tile kernels' loops from being unrolled.
static __device__ __attribute__((noinline)) float2 rope_sincos_large(float theta) {
    float x;
    int quad;
    rope_reduce_large(theta, x, quad);
    float2 sc;
    rope_sincos_reduced(x, quad, sc.x, sc.y);
    return sc;
}

// Sine and cosine of a float32 angle.  The angle is reduced by the nearest multiple of pi/2 in double (an error below
// 10^-9 up to 2^24), the remainder goes through the Taylor polynomials of degree 9 and 10 (next terms below 2 10^-9 and
// 2 10^-10 there): against float64, rotated float32 rows at positions up to 10^6 are off by 4.4 10^-8 (2-norm), by
// 4.5 10^-8 with the library's sincosf.  Some 30 instructions; sincosf carries a multi-word reduction for large angles
// that the appends spent most of their time in (512 rows of 8 heads x 128: 22.7 us full precision and 18.8 us quantized
// with it and an exponential per element, 10.3 and 11.4 us so).
constexpr float ROPE_LARGE = 16777216.f;
__device__ __forceinline__ void rope_reduce(float theta, float &x, int &quad) {
    const double t = (double)theta;
    const double k = rint(t * 0.63661977236758134308);
    x = (float)fma(-k, 1.57079632679489661923, t);
    quad = (int)(k - 4.0 * floor(k * 0.25));
}
// (CALL: in code that is repeated for many elements)
template <bool CALL>
__device__ __forceinline__ void rope_sincos(float theta, float &sn, float &cs) {
    float x;
    int quad;
    rope_reduce(theta, x, quad);
    if (!CALL && __builtin_expect(fabsf(theta) >= ROPE_LARGE, 0)) rope_reduce_large(theta, x, quad);
    rope_sincos_reduced(x, quad, sn, cs);
    if (CALL && __builtin_expect(fabsf(theta) >= ROPE_LARGE, 0)) {
        const float2 sc = rope_sincos_large(theta);
        sn = sc.x;
        cs = sc.y;
    }
}
// The same for V angles, with one look at the largest (512 rows of 8 heads x 128 at 4 bits, the rotated append: 11.8 us;
// 13.3 with a branch behind each angle, 11.0 with none).
template <int V, class ANGLE>
__device__ __forceinline__ void rope_sincos_many(ANGLE angle, float (&sn)[V], float (&cs)[V]) {
    float largest = 0.f;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const float theta = angle(j);
        largest = fmaxf(largest, fabsf(theta));
        float x;
        int quad;
        rope_reduce(theta, x, quad);
        rope_sincos_reduced(x, quad, sn[j], cs[j]);
    }
    if (__builtin_expect(largest >= ROPE_LARGE, 0)) {
#pragma unroll 1
        for (int i = 0; i < V; ++i) {
            const float theta = angle(i);
            if (fabsf(theta) < ROPE_LARGE) continue;
            const float2 sc = rope_sincos_large(theta);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                sn[j] = j == i ? sc.x : sn[j];
                cs[j] = j == i ? sc.y : cs[j];
            }
        }
    }
}

// The inverse frequency of pair i is formed in double and rounded once, so that it does not depend on
// one exp implementation's last float32 bit (a position of 10^5 turns one such bit into 10^-2 rad).
__device__ __forceinline__ float rope_inv_freq(const RopeDev &r, int i) {
    return r.freqs ? 1.0f / r.freqs[i] : (float)exp(-(double)i * r.log_base_over_half);
}
__device__ __forceinline__ float rope_angle(const RopeDev &r, int pos, float inv) { return ((float)pos * r.scale) * inv; }
__device__ __forceinline__ int rope_pos(const RopeDev &r, int bh, int l) {
    return (r.batch_pos ? r.batch_pos[bh / r.H] : r.pos0) + l;
}
// one element of a rotated pair (x: itself, y: its partner)
__device__ __forceinline__ float rope_turn(float x, float y, bool first, float sn, float cs) {
    return first ? x * cs - y * sn : y * sn + x * cs;
}

// Element d of a row at position `pos` after the rotary embedding, rounded to the row's dtype
// (what the reference hands to the cache: `applyRotaryPosition` runs before `update`,
// Llama.swift:58-62).  The angle is the float32 product of position * scale and the inverse
// frequency exp(-i * log(base) / half), or 1 / freqs[i].
template <int DT, bool CALL = false>
__device__ __forceinline__ float rope_elem(const RopeDev &r, const void *row, int d, int pos) {
    const float x = Elem<DT>::load(row, d);
    if (d >= r.dims) return x;
    const int half = r.dims >> 1;
    int i, partner;
    bool first;
    if (r.traditional) {
        i = d >> 1;
        partner = d ^ 1;
        first = (d & 1) == 0;
    } else {
        first = d < half;
        i = first ? d : d - half;
        partner = first ? d + half : d - half;
    }
    float sn, cs;
    rope_sincos<CALL>(rope_angle(r, pos, rope_inv_freq(r, i)), sn, cs);
    return round_dt<DT>(rope_turn(x, Elem<DT>::load(row, partner), first, sn, cs));
}

// ---- 16-byte chunks: V = 8 elements of a 16-bit dtype, 4 floats ------------------------------------------------
// (RopeDev::vec says that pairs never cut through a chunk)
template <int DT> constexpr int rope_chunk_elems() { return DT == 2 ? 4 : 8; }
template <int DT> __device__ __forceinline__ void chunk_unpack(const kv_u4 &raw, float (&w)[rope_chunk_elems<DT>()]) {
    const uint32_t u[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (DT == 2) {
            w[j] = __uint_as_float(u[j]);
        } else if constexpr (DT == 1) {
            w[2 * j] = __uint_as_float(u[j] << 16);
            w[2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u);
        } else {
            w[2 * j] = __half2float(__ushort_as_half((unsigned short)(u[j] & 0xffffu)));
            w[2 * j + 1] = __half2float(__ushort_as_half((unsigned short)(u[j] >> 16)));
        }
    }
}
template <int DT> __device__ __forceinline__ kv_u4 chunk_pack(const float (&w)[rope_chunk_elems<DT>()]) {
    uint32_t u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (DT == 2) u[j] = __float_as_uint(w[j]);
        else if constexpr (DT == 1) u[j] = (uint32_t)Elem<1>::bits(w[2 * j]) | ((uint32_t)Elem<1>::bits(w[2 * j + 1]) << 16);
        else u[j] = (uint32_t)__half_as_ushort(__float2half_rn(w[2 * j])) | ((uint32_t)__half_as_ushort(__float2half_rn(w[2 * j + 1])) << 16);
    }
    return kv_u4{u[0], u[1], u[2], u[3]};
}
// the inverse frequencies of all pairs, into LDS (the caller synchronises)
__device__ __forceinline__ void rope_inv_table(const RopeDev &r, float *inv_s) {
    for (int i = threadIdx.x; i < (r.dims >> 1); i += blockDim.x) inv_s[i] = rope_inv_freq(r, i);
}
// sines and cosines for the elements of the chunk at d0 < dims (one per pair: `traditional` chunks hold V / 2 pairs)
template <int DT>
__device__ __forceinline__ void rope_chunk_sincos(const RopeDev &r, const float *inv_s, int d0, int pos,
                                                  float (&sn)[rope_chunk_elems<DT>()], float (&cs)[rope_chunk_elems<DT>()]) {
    constexpr int V = rope_chunk_elems<DT>();
    if (r.traditional) {
        float s[V / 2], c[V / 2];
        rope_sincos_many<V / 2>([&](int j) { return rope_angle(r, pos, inv_s[d0 / 2 + j]); }, s, c);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            sn[j] = s[j / 2];
            cs[j] = c[j / 2];
        }
    } else {
        const int half = r.dims >> 1, i0 = d0 < half ? d0 : d0 - half;
        rope_sincos_many<V>([&](int j) { return rope_angle(r, pos, inv_s[i0 + j]); }, sn, cs);
    }
}
// The chunk at d0 < dims of a row, rotated and rounded to the dtype; `row` is the unrotated row.
template <int DT>
__device__ __forceinline__ void rope_chunk(const RopeDev &r, const float *inv_s, const char *row, int d0, int pos, const kv_u4 &raw,
                                           float (&w)[rope_chunk_elems<DT>()]) {
    constexpr int V = rope_chunk_elems<DT>();
    const int half = r.dims >> 1;
    const bool first = d0 < half;
    float x[V], y[V], sn[V], cs[V];
    chunk_unpack<DT>(raw, x);
    if (!r.traditional)
        chunk_unpack<DT>(*reinterpret_cast<const kv_u4 *>(row + (size_t)(first ? d0 + half : d0 - half) * (DT == 2 ? 4 : 2)), y);
    rope_chunk_sincos<DT>(r, inv_s, d0, pos, sn, cs);
#pragma unroll
    for (int j = 0; j < V; ++j)
        w[j] = round_dt<DT>(r.traditional ? rope_turn(x[j], x[j ^ 1], (j & 1) == 0, sn[j], cs[j]) : rope_turn(x[j], y[j], first, sn[j], cs[j]));
}

// ---- one token's rows, for the decode kernels --------------------------------------------------------------------
// The R query rows (adjacent, D elements) and the key row of one kv head, rotated and rounded to the dtype, into LDS
// [R + 1][D]; the caller synchronises.  A thread owns one pair of columns and forms its sine and cosine once; all THREADS
// threads of the workgroup take part.  Every workgroup of the launch does this for itself, where a launch for it takes 4 to
// 6.5 us.  In two halves: `fetch` requests the elements (of at most RMAX query rows) in front of the workgroup's first key
// loads -- loads complete in order --, `turn` works the angles out and turns the rows while those keys are on their way.
template <int DT, int D, int THREADS, int RMAX> struct RopeStep {
    static constexpr int P = D / 2, NS = THREADS / P, NR = (RMAX + 1 + NS - 1) / NS;  // pairs of a row; rows at once; rows of a thread
    static_assert(NS >= 1, "a thread per pair of columns");
    int d0, d1;
    bool rotates;
    float freq;
    using E = typename Elem<DT>::type;
    E x[NR], y[NR];
    // Row J * NS and on of a thread.  (One row at a time: a uniform number, and a wavefront does not run through the code of
    // rows that there are not.)
    template <int J> __device__ __forceinline__ void fetch_rows(const E *q, const E *k, int R) {
        if constexpr (J < NR) {
            const int i = (NS == 1 ? 0 : threadIdx.x / P) + J * NS;
            if (NS == 1 && i > R) return;
            if (i <= R && (NS * P == THREADS || threadIdx.x < NS * P)) {
                const E *row = i < R ? q + (size_t)i * D : k;
                x[J] = row[d0];
                y[J] = row[d1];
            }
            fetch_rows<J + 1>(q, k, R);
        }
    }
    template <int J> __device__ __forceinline__ void turn_rows(float sn, float cs, int R, E *dst) {
        if constexpr (J < NR) {
            const int i = (NS == 1 ? 0 : threadIdx.x / P) + J * NS;
            if (NS == 1 && i > R) return;
            if (i <= R && (NS * P == THREADS || threadIdx.x < NS * P)) {
                if (rotates) {
                    const float a = Elem<DT>::load(&x[J], 0), b = Elem<DT>::load(&y[J], 0);
                    Elem<DT>::store(&x[J], 0, rope_turn(a, b, true, sn, cs));
                    Elem<DT>::store(&y[J], 0, rope_turn(b, a, false, sn, cs));
                }
                dst[i * D + d0] = x[J];
                dst[i * D + d1] = y[J];
            }
            turn_rows<J + 1>(sn, cs, R, dst);
        }
    }
    __device__ __forceinline__ void fetch(const RopeDev &r, const E *q, const E *k, int R) {
        const int p = threadIdx.x % P, half = r.dims >> 1;
        rotates = p < half;
        d0 = !rotates ? r.dims + 2 * (p - half) : r.traditional ? 2 * p : p;
        d1 = rotates && !r.traditional ? d0 + half : d0 + 1;
        freq = 1.f;
        if (r.freqs && rotates) freq = r.freqs[p];
        fetch_rows<0>(q, k, R);
    }
    __device__ __forceinline__ void turn(const RopeDev &r, int bh, int R, E *dst) {
        float sn = 0.f, cs = 1.f;
        if (rotates) {
            const float inv = r.freqs ? 1.0f / freq : (float)exp(-(double)(int)(threadIdx.x % P) * r.log_base_over_half);
            rope_sincos<false>(rope_angle(r, rope_pos(r, bh, 0), inv), sn, cs);
        }
        // (`freq` lives to here: its register holds what may be a load in flight, and the angle, formed in it, would wait for
        // every load requested since, the first tile's with them)
        asm volatile("" ::"v"(freq));
        turn_rows<0>(sn, cs, R, dst);
    }
};

// ---- the queries of a forward ----------------------------------------------------------------------------------
// Threads of a workgroup that turn queries.
__host__ __device__ __forceinline__ int rope_ride_threads(int block) { return block < 256 ? block : 256; }
// One row position (batch row b, row l of L) of `x` [B, H, L, D] into `out` (which may be x) for heads [h0, h1): a
// thread owns one chunk pair (chunk, when the pairs are adjacent), works out its sines and cosines once and turns
// that chunk pair of every head it takes.  `inv_s`: dims / 2 floats of LDS.  Workgroups of any width that holds a head's
// items (the appends' are 192, 256 and 512 wide; of 512 threads the first 256 work).
// Bound by the read and the write of the queries: 512 rows of 32 heads x 128 in bfloat16, 8.4 MB, see
// rope_rows_kernel.
template <int DT>
__device__ __forceinline__ void rope_rows_body(const RopeDev &r, const char *x, char *out, int H, int L, int D, int b, int l,
                                               int h0, int h1, float *inv_s) {
    constexpr int V = rope_chunk_elems<DT>(), ES = DT == 2 ? 4 : 2;
    const int half = r.dims >> 1;
    const int np = r.traditional ? r.dims / V : half / V;  // rotating items of a head, then the chunks that pass through
    const int items = np + (D - r.dims) / V;
    int slot, ns;  // (the usual numbers of items without a division: the first loads wait for these)
    if (__builtin_expect((items & (items - 1)) == 0, 1)) {
        const int sh = 31 - __clz(items);
        slot = threadIdx.x >> sh;
        ns = rope_ride_threads((int)blockDim.x) >> sh;
    } else {
        slot = threadIdx.x / items;
        ns = rope_ride_threads((int)blockDim.x) / items;
    }
    const int item = threadIdx.x - slot * items;
    const bool live = slot < ns;
    const bool turn = item < np;
    const int d0 = turn ? item * V : r.dims + (item - np) * V;
    const int d1 = turn && !r.traditional ? d0 + half : d0;
    const size_t hs = (size_t)L * D * ES;
    const size_t off = ((size_t)b * H * L + l) * D * ES;
    int h = h0 + slot;
    kv_u4 a{0u, 0u, 0u, 0u}, c{0u, 0u, 0u, 0u};
    const bool some = live && h < h1;
    if (some) {
        a = *reinterpret_cast<const kv_u4 *>(x + off + h * hs + (size_t)d0 * ES);
        c = *reinterpret_cast<const kv_u4 *>(x + off + h * hs + (size_t)d1 * ES);
    }
    rope_inv_table(r, inv_s);
    __syncthreads();
    if (!some) return;
    float sn[V], cs[V];
    if (turn) rope_chunk_sincos<DT>(r, inv_s, d0, (r.batch_pos ? r.batch_pos[b] : r.pos0) + l, sn, cs);
    for (;;) {
        const int hn = h + ns;
        kv_u4 an = a, cn = c;
        if (hn < h1) {
            an = *reinterpret_cast<const kv_u4 *>(x + off + hn * hs + (size_t)d0 * ES);
            cn = *reinterpret_cast<const kv_u4 *>(x + off + hn * hs + (size_t)d1 * ES);
        }
        if (turn) {
            float xa[V], xc[V], ya[V], yc[V];
            chunk_unpack<DT>(a, xa);
            chunk_unpack<DT>(c, xc);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                if (r.traditional) {
                    ya[j] = rope_turn(xa[j], xa[j ^ 1], (j & 1) == 0, sn[j], cs[j]);
                } else {
                    ya[j] = rope_turn(xa[j], xc[j], true, sn[j], cs[j]);
                    yc[j] = rope_turn(xc[j], xa[j], false, sn[j], cs[j]);
                }
            }
            a = chunk_pack<DT>(ya);
            if (!r.traditional) *reinterpret_cast<kv_u4 *>(out + off + h * hs + (size_t)d1 * ES) = chunk_pack<DT>(yc);
        }
        *reinterpret_cast<kv_u4 *>(out + off + h * hs + (size_t)d0 * ES) = a;
        if (hn >= h1) return;
        h = hn;
        a = an;
        c = cn;
    }
}

// Heads one workgroup of the query pass takes: all of them where the row positions fill the chip, and otherwise as many
// as its threads turn at once, so that none of them walks heads one after the other behind its exponentials.
// (64 heads x 128, one token, batch 8, with a workgroup per batch row: 4.75 us, against 4.2 us in workgroups of 32 heads.)
__host__ __device__ __forceinline__ int rope_heads_per_group(int rows, int H, int D, int es, int block) {
    if (rows >= 256) return H;
    const int at_once = rope_ride_threads(block) / max(1, D * es / 32);  // 32 bytes, a chunk pair, per thread
    return min(H, max(1, at_once));
}
// The query workgroups behind the `bh` rows of an append's grid (blockIdx.y >= bh): workgroup number i of them takes
// the heads of group i % groups at row position i / groups.
template <int DT>
__device__ __forceinline__ void rope_queries_ride(const RopeDev &r, int bh, float *inv_s) {
    const int i = (blockIdx.y - bh) * gridDim.x + blockIdx.x, rows = r.qB * r.qL;
    const int hg = rope_heads_per_group(rows, r.qH, r.qD, DT == 2 ? 4 : 2, (int)blockDim.x);
    int row = i, h0 = 0, b = 0;
    if (hg < r.qH) {
        const int groups = (r.qH + hg - 1) / hg;
        row = i / groups;
        h0 = (i - row * groups) * hg;
    }
    if (row >= rows) return;
    if (r.qB > 1) b = row / r.qL;
    rope_rows_body<DT>(r, r.qx, r.qo, r.qH, r.qL, r.qD, b, row - b * r.qL, h0, min(r.qH, h0 + hg), inv_s);
}
// Rows those workgroups add to the grid of an append whose rows are `gx` workgroups of `block` threads wide; 0: none ride.
inline int rope_ride_rows(const RopeDev &r, int gx, int es, int block) {
    if (r.qx == nullptr) return 0;
    const int rows = r.qB * r.qL, hg = rope_heads_per_group(rows, r.qH, r.qD, es, block);
    return (int)(((long)rows * ((r.qH + hg - 1) / hg) + gx - 1) / gx);
}

}  // namespace kvhip
