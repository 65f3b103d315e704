// Append (full precision and quantize-on-append), import/export between the
// page layout and the reference's dense array layout, ring-order gather, and
// the standalone affine quantizer.
#include "kvhip_quant_tile.hpp"

namespace kvhip {

namespace {

// grid (L, B, head groups): the queries of one row position (rope_rows_body).  512 rows of 32 heads x 128 in
// bfloat16 (8.4 MB moved): 10.5 us with a workgroup per row and head and a sine, cosine and exponential per element,
// 4.9 us so.
template <int DT>
__global__ void __launch_bounds__(256) rope_rows_kernel(RopeDev r, const char *x, char *out, int H, int L, int D) {
    __shared__ float inv_s[512];
    const int hg = rope_heads_per_group(gridDim.x * gridDim.y, H, D, DT == 2 ? 4 : 2, 256), h0 = blockIdx.z * hg;
    rope_rows_body<DT>(r, x, out, H, L, D, blockIdx.y, blockIdx.x, h0, min(H, h0 + hg), inv_s);
}

// grid (L, B*H): one row per workgroup; arrays whose pairs cut through 16-byte chunks
template <int DT>
__global__ void rope_apply_kernel(RopeDev r, const char *x, char *out, int L, int D) {
    const int bh = blockIdx.y, l = blockIdx.x;
    const size_t off = ((size_t)bh * L + l) * D * (DT == 2 ? 4 : 2);
    const int pos = rope_pos(r, bh, l);
    // every element is read (with its partner) before any is written: out may alias x
    float v[4];
    int cnt = 0;
    for (int d = threadIdx.x; d < D; d += blockDim.x) v[cnt++] = rope_elem<DT>(r, x + off, d, pos);
    __syncthreads();
    cnt = 0;
    for (int d = threadIdx.x; d < D; d += blockDim.x) Elem<DT>::store(out + off, d, v[cnt++]);
}

// One wavefront quantizes one row of D elements.  Optional outputs:
//   k_words   packed codes in MLX order (D*BITS/32 words)
//   code_out  one byte per element (for the transposed V assembly)
//   sb_row    (scale,bias) pairs of dtype DT per group
//   scales/biases separate arrays of dtype DT per group
template <int DT, int BITS>
__device__ __forceinline__ void quantize_row_wave(const void *src, int D, int gs, int lane,
                                                  uint32_t *k_words, uint8_t *code_out, void *sb_row,
                                                  void *scales, void *biases, const RopeDev *rope = nullptr,
                                                  int pos = 0) {
    quantize_row_wave_from<DT, BITS>(
        [&](int d) { return rope ? rope_elem<DT>(*rope, src, d, pos) : Elem<DT>::load(src, d); }, D, gs, lane, k_words,
        [&](int d, uint32_t code) { if (code_out) code_out[d] = (uint8_t)code; }, sb_row, scales, biases);
}

// grid (rows, BH + query rows): one new row per workgroup, scattered into the chunk-interleaved tile; RIDE: with queries
// of the same forward behind them (RopeDev::qx; 256 threads then).
template <int ES, bool RIDE>
__global__ void append_fp_kernel(Store st, const char *keys, const char *values, int L, int src0,
                                 int slot0, RopeDev rope) {
    const int bh = blockIdx.y;
    if constexpr (RIDE) {
        if (bh >= st.BH) {
            __shared__ float inv_s[512];
            if (ES == 4) rope_queries_ride<2>(rope, st.BH, inv_s);
            else if (st.dtype == KVHIP_F16) rope_queries_ride<0>(rope, st.BH, inv_s);
            else rope_queries_ride<1>(rope, st.BH, inv_s);
            return;
        }
    }
    const int i = blockIdx.x;
    const int slot = slot0 + i;
    const int l = src0 + i;
    using E = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
    const E *ks = reinterpret_cast<const E *>(keys) + ((size_t)bh * L + l) * st.Dk;
    char *kc = const_cast<char *>(k_cell_ptr(st, bh, slot));
    if (rope.dims > 0) {
        const int pos = rope_pos(rope, bh, l);
        for (int d = threadIdx.x; d < st.Dk; d += blockDim.x) {
            char *dst = kc + kfp_off(st, slot, d);
            if (ES == 4) Elem<2>::store(dst, 0, rope_elem<2>(rope, ks, d, pos));
            else if (st.dtype == KVHIP_F16) Elem<0>::store(dst, 0, rope_elem<0>(rope, ks, d, pos));
            else Elem<1>::store(dst, 0, rope_elem<1>(rope, ks, d, pos));
        }
    } else {
        for (int d = threadIdx.x; d < st.Dk; d += blockDim.x) *reinterpret_cast<E *>(kc + kfp_off(st, slot, d)) = ks[d];
    }
    const E *vs = reinterpret_cast<const E *>(values) + ((size_t)bh * L + l) * st.Dv;
    char *vc = const_cast<char *>(v_cell_ptr(st, bh, slot));
    for (int d = threadIdx.x; d < st.Dv; d += blockDim.x) *reinterpret_cast<E *>(vc + vfp_off(st, slot, d)) = vs[d];
}

// grid (64-token tiles touched, BH), 256 threads.  Each wavefront quantizes rows of
// the tile; V codes are staged as bytes in LDS and then merged into the transposed
// tile rows, touching only the token positions this append writes.
// (ROPE = false carries no rotation code: the single-token decode append stays as small as it was)
// PAGED: the new rows are rows [src0, src0 + n) of the full-precision page store `src` (a cache
// being converted) instead of dense arrays.
template <int DT, int BITS, bool ROPE, bool PAGED>
__device__ __forceinline__ void append_quant_body(const Store &st, const Store &src, const char *keys, const char *values,
                                                  int L, int src0, int slot0, int n, const RopeDev &rope) {
    extern __shared__ __attribute__((aligned(16))) uint8_t vcodes[];  // [64][Dv]
    const int bh = blockIdx.y;
    const int tile = (slot0 >> 6) + blockIdx.x;
    const int lo = max(slot0, tile * TILE);
    const int hi = min(slot0 + n, tile * TILE + TILE);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    constexpr int TPW = 32 / BITS;          // tokens per word
    const int t_lo = lo & (TILE - 1), t_hi = t_lo + (hi - lo);
    // the words of a V tile row this append touches, and this thread's first merge item:
    // its old word is requested now, so a single-token append does not wait for it later
    // (for 3, 5 and 6 bits a token's code may straddle two words of the row's bit stream)
    const int w_lo = (t_lo * BITS) >> 5, nw = ((t_hi * BITS - 1) >> 5) - w_lo + 1;
    const int items = st.Dv * nw;
    char *cell = const_cast<char *>(v_cell_ptr(st, bh, lo));
    auto word_ptr = [&](int u) -> uint32_t * {
        const int d = u / nw, w = w_lo + (u - d * nw);
        return reinterpret_cast<uint32_t *>(cell + v_row_off(st, lo, d)) + w;
    };
    const bool partial = ((t_lo * BITS) & 31) != 0 || ((t_hi * BITS) & 31) != 0;  // some word keeps old tokens
    uint32_t old0 = 0;
    if (partial && (int)threadIdx.x < items) old0 = *word_ptr(threadIdx.x);
    // (row, K or V) pairs go round the wavefronts (four, or eight for appends of three rows and more), so one
    // new token uses two of them
    const int nwaves = blockDim.x >> 6;
    for (int item = wave; item < 2 * (hi - lo); item += nwaves) {
        const int slot = lo + (item >> 1);
        const int l = src0 + (slot - slot0);
        uint32_t *kw = reinterpret_cast<uint32_t *>(const_cast<char *>(k_row_ptr(st, bh, slot)));
        if constexpr (PAGED) {
            if ((item & 1) == 0) {
                const char *kc = k_cell_ptr(src, bh, l);
                quantize_row_wave_from<DT, BITS>([&](int d) { return Elem<DT>::load(kc + kfp_off(src, l, d), 0); }, st.Dk, st.gs,
                                                 lane, kw, [](int, uint32_t) {}, const_cast<char *>(ksb_row_ptr(st, bh, slot)),
                                                 nullptr, nullptr);
            } else {
                const char *vc = v_cell_ptr(src, bh, l);
                uint8_t *vc_out = vcodes + (slot & (TILE - 1)) * st.Dv;
                quantize_row_wave_from<DT, BITS>([&](int d) { return Elem<DT>::load(vc + vfp_off(src, l, d), 0); }, st.Dv, st.gs,
                                                 lane, nullptr, [&](int d, uint32_t code) { vc_out[d] = (uint8_t)code; },
                                                 const_cast<char *>(vsb_row_ptr(st, bh, slot)), nullptr, nullptr);
            }
        } else if ((item & 1) == 0) {
            const char *krow = keys + ((size_t)bh * L + l) * st.Dk * st.es;
            quantize_row_wave<DT, BITS>(krow, st.Dk, st.gs, lane, kw, nullptr, const_cast<char *>(ksb_row_ptr(st, bh, slot)),
                                        nullptr, nullptr, ROPE ? &rope : nullptr, ROPE ? rope_pos(rope, bh, l) : 0);
        } else {
            const char *vrow = values + ((size_t)bh * L + l) * st.Dv * st.es;
            quantize_row_wave<DT, BITS>(vrow, st.Dv, st.gs, lane, nullptr, vcodes + (slot & (TILE - 1)) * st.Dv,
                                        const_cast<char *>(vsb_row_ptr(st, bh, slot)), nullptr, nullptr);
        }
    }
    __syncthreads();
    for (int u = threadIdx.x; u < items; u += blockDim.x) {
        const int d = u / nw, w = w_lo + (u - d * nw);
        uint32_t nbits = 0, mbits = 0;
        if constexpr ((32 % BITS) == 0) {
            for (int tt = 0; tt < TPW; ++tt) {
                const int t = w * TPW + tt;
                if (t >= t_lo && t < t_hi) {
                    const int bp = v_bitpos<BITS>(t) & 31;
                    nbits |= (uint32_t)vcodes[t * st.Dv + d] << bp;
                    mbits |= ((1u << BITS) - 1u) << bp;
                }
            }
        } else {
            const int t0 = (32 * w) / BITS;  // the first token with bits in word w
            for (int tt = 0; tt < TPW + 2; ++tt) {
                const int t = t0 + tt;
                if (t >= t_lo && t < t_hi && t * BITS < 32 * w + 32) {
                    nbits |= stream_bits(vcodes[t * st.Dv + d], t * BITS, w);
                    mbits |= stream_bits((1u << BITS) - 1u, t * BITS, w);
                }
            }
        }
        uint32_t *p = word_ptr(u);
        if (mbits == 0xffffffffu) {
            *p = nbits;
        } else {
            const uint32_t old = (u == (int)threadIdx.x) ? old0 : *p;
            *p = (old & ~mbits) | nbits;
        }
    }
}

// grid (64-token tiles touched, BH), 256 threads.  Each wavefront quantizes rows of
// the tile; V codes are staged as bytes in LDS and then merged into the transposed
// tile rows, touching only the token positions this append writes.
// (ROPE = false carries no rotation code: the single-token decode append stays as small as it was)
template <int DT, int BITS, bool ROPE>
__global__ void __launch_bounds__(512)
append_quant_kernel(Store st, const char *keys, const char *values, int L, int src0, int slot0, int n,
                    RopeDev rope) {
    if constexpr (ROPE) {
        if ((int)blockIdx.y >= st.BH) {  // queries of the same forward (64 Dv bytes of LDS hold dims / 2 floats)
            extern __shared__ __attribute__((aligned(16))) uint8_t vcodes[];
            rope_queries_ride<DT>(rope, st.BH, reinterpret_cast<float *>(vcodes));
            return;
        }
    }
    append_quant_body<DT, BITS, ROPE, false>(st, st, keys, values, L, src0, slot0, n, rope);
}

// The same for rows [row0, row0 + n) of a full-precision page store, written to the same slots of `st`.
template <int DT, int BITS>
__global__ void __launch_bounds__(256) requant_rows_kernel(Store st, Store src, int row0, int n) {
    append_quant_body<DT, BITS, false, true>(st, src, nullptr, nullptr, 0, row0, row0, n, RopeDev());
}


// grid (64-token tiles, BH): rows [0, rows) of a quantized store as full-precision rows of `dst`
// (`MLX.dequantized`: scale * code + bias in float32, rounded once to the dtype)
template <int DT, int BITS>
__global__ void __launch_bounds__(256) dequant_pages_kernel(Store q, Store dst, int rows) {
    const int bh = blockIdx.y;
    const int lo = blockIdx.x * TILE, hi = min(rows, lo + TILE);
    for (int idx = threadIdx.x; idx < (hi - lo) * q.Dk; idx += 256) {
        const int t = idx / q.Dk, d = idx - t * q.Dk, slot = lo + t;
        const uint32_t c = stream_code<BITS>(reinterpret_cast<const uint32_t *>(k_row_ptr(q, bh, slot)), d);
        const char *sb = ksb_row_ptr(q, bh, slot);
        const float sc = Elem<DT>::load(sb, 2 * (d / q.gs)), bi = Elem<DT>::load(sb, 2 * (d / q.gs) + 1);
        Elem<DT>::store(const_cast<char *>(k_cell_ptr(dst, bh, slot)) + kfp_off(dst, slot, d), 0, __fadd_rn(__fmul_rn(sc, (float)c), bi));
    }
    const char *vcell = v_cell_ptr(q, bh, lo);
    for (int idx = threadIdx.x; idx < (hi - lo) * q.Dv; idx += 256) {
        const int d = idx / (hi - lo), t = idx - d * (hi - lo), slot = lo + t;   // consecutive threads: consecutive tokens of a column
        const uint32_t c = v_code_load<BITS>(vcell + v_row_off(q, lo, d), t);
        const char *sb = vsb_row_ptr(q, bh, slot);
        const float sc = Elem<DT>::load(sb, 2 * (d / q.gs)), bi = Elem<DT>::load(sb, 2 * (d / q.gs) + 1);
        Elem<DT>::store(const_cast<char *>(v_cell_ptr(dst, bh, slot)) + vfp_off(dst, slot, d), 0, __fadd_rn(__fmul_rn(sc, (float)c), bi));
    }
}

// The same for 16-bit dtypes and head sizes that are multiples of 8, in whole tiles and 16-byte pieces: a thread forms
// eight adjacent elements of a K row, or one column's values for eight adjacent tokens, which is one 16-byte chunk of
// the interleaved full-precision tile; consecutive threads write consecutive chunks.  grid (tiles, BH, 2): K and V of a
// tile are separate workgroups; a thread requests the codes and (scale, bias) pairs of up to four chunks before it
// converts the first.  Eight codes lie inside two adjacent dwords for every code width (a V tile row's octet of
// tokens likewise, in the order v_bitpos gives).  Rows past the cache's length in the last tile come out as
// whatever their slots hold (zeros, or rows trimmed earlier): finite values nobody presents.
template <int DT> __device__ __forceinline__ void pair_of(uint32_t raw, float &sc, float &bi) {
    if (DT == 0) {
        sc = (float)__builtin_bit_cast(_Float16, (uint16_t)raw);
        bi = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw >> 16));
    } else {
        sc = __uint_as_float(raw << 16);
        bi = __uint_as_float(raw & 0xffff0000u);
    }
}
// `dst_pt` non-null: the destination is scratch whose page p lies at `page0` + p * (sk, sv) and whose page table
// `dst_pt` is still unwritten -- the first workgroup writes its `pages` entries for the kernels that follow, and
// nobody here reads them.
template <int DT, int BITS>
__global__ void __launch_bounds__(256) dequant_tiles16_kernel(Store q, Store dst, PageEntry *dst_pt, int pages, PageEntry page0, size_t sk, size_t sv) {
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    constexpr uint32_t M = (1u << BITS) - 1u;
    constexpr int NB = 4;  // chunks in flight per thread
    const int bh = blockIdx.y, lo = blockIdx.x * TILE;
    auto pack = [](float a, float b) { return DT == 0 ? pk_h2(a, b) : pk_bf2(a, b); };
    if (dst_pt != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) {
        for (int p = threadIdx.x; p < pages; p += 256) {
            PageEntry e;
            e.k = page0.k + (size_t)p * sk;
            e.v = page0.v + (size_t)p * sv;
            dst_pt[p] = e;
        }
    }
    const PageEntry de = dst_pt != nullptr ? PageEntry{page0.k + (size_t)(lo >> PAGE_SHIFT) * sk, nullptr, page0.v + (size_t)(lo >> PAGE_SHIFT) * sv, nullptr}
                                           : dst.pt[lo >> PAGE_SHIFT];
    if (blockIdx.z == 0) {
        char *kdst = de.k + (size_t)bh * dst.k_cell + kfp_off(dst, lo, 0);
        const int items = (q.Dk / 8) * TILE, last = (int)q.k_row / 4 - 1;
        for (int base = threadIdx.x; base < items; base += 256 * NB) {
            uint32_t w0[NB], w1[NB], sb[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int item = base + 256 * u;
                if (item < items) {
                    const int c = item >> 6, slot = lo + (item & 63), wi = (8 * c * BITS) >> 5;
                    const uint32_t *row = reinterpret_cast<const uint32_t *>(k_row_ptr(q, bh, slot));
                    w0[u] = row[wi];
                    w1[u] = row[min(wi + 1, last)];
                    sb[u] = reinterpret_cast<const uint32_t *>(ksb_row_ptr(q, bh, slot))[(8 * c) / q.gs];
                }
            }
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int item = base + 256 * u;
                if (item < items) {
                    const int off = ((item >> 6) * 8 * BITS) & 31;
                    const uint64_t bits = (((uint64_t)w1[u] << 32) | w0[u]) >> off;
                    float sc, bi, x[8];
                    pair_of<DT>(sb[u], sc, bi);
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[j] = __fadd_rn(__fmul_rn(sc, (float)((uint32_t)(bits >> (j * BITS)) & M)), bi);
                    *reinterpret_cast<u4v *>(kdst + (size_t)item * 16) = u4v{pack(x[0], x[1]), pack(x[2], x[3]), pack(x[4], x[5]), pack(x[6], x[7])};
                }
            }
        }
        return;
    }
    const char *vcell = v_cell_ptr(q, bh, lo);
    char *vdst = de.v + (size_t)bh * dst.v_cell + vfp_off(dst, lo, 0);
    const int items = 8 * q.Dv, last = TILE * BITS / 32 - 1;
    for (int base = threadIdx.x; base < items; base += 256 * NB) {
        uint32_t w0[NB], w1[NB], sb[NB][8];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int item = base + 256 * u;
            if (item < items) {
                const int tc = item / q.Dv, d = item - tc * q.Dv, wi = v_bitpos<BITS>(8 * tc) >> 5;
                const uint32_t *row = reinterpret_cast<const uint32_t *>(vcell + v_row_off(q, lo, d));
                w0[u] = row[wi];
                w1[u] = row[min(wi + 1, last)];
                const int g = d / q.gs;
#pragma unroll
                for (int j = 0; j < 8; ++j) sb[u][j] = reinterpret_cast<const uint32_t *>(vsb_row_ptr(q, bh, lo + 8 * tc + j))[g];
            }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int item = base + 256 * u;
            if (item < items) {
                const int tc = item / q.Dv, first = v_bitpos<BITS>(8 * tc) & ~31;
                const uint64_t bits = ((uint64_t)w1[u] << 32) | w0[u];
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float sc, bi;
                    pair_of<DT>(sb[u][j], sc, bi);
                    x[j] = __fadd_rn(__fmul_rn(sc, (float)((uint32_t)(bits >> (v_bitpos<BITS>(8 * tc + j) - first)) & M)), bi);
                }
                *reinterpret_cast<u4v *>(vdst + (size_t)item * 16) = u4v{pack(x[0], x[1]), pack(x[2], x[3]), pack(x[4], x[5]), pack(x[6], x[7])};
            }
        }
    }
}

// The same for head sizes that are multiples of 32, by units of 32 codes (4 BITS bytes: whole dwords for every code
// width).  A thread loads one unit -- the units of a tile's K rows, and of its V tile rows, are one contiguous run, so
// the loads of a workgroup are too --, converts it and writes four 16-byte chunks of the interleaved full-precision
// tile; for each of the four, the threads of a wavefront write runs of 256 bytes (K: sixteen tokens of one chunk
// column) or 512 bytes (V: thirty-two columns of one token octet).  A K unit has one (scale, bias) pair, loaded with
// it; a V unit needs the pairs of its 32 tokens, which the workgroup stages in LDS once ([group][token]).
// code j (0..31) of a unit held in N dwords, at unit-relative bit `pos` (constant once unrolled)
template <int BITS, int N> __device__ __forceinline__ uint32_t unit_code(const uint32_t (&w)[N], int pos) {
    const int wi = pos >> 5, sh = pos & 31;
    uint32_t v = w[wi] >> sh;
    if (sh + BITS > 32) v |= w[wi + 1 < N ? wi + 1 : wi] << ((32 - sh) & 31);
    return v & ((1u << BITS) - 1u);
}
template <int DT, int BITS>
__global__ void __launch_bounds__(256) dequant_units_kernel(Store q, Store dst, PageEntry *dst_pt, int pages, PageEntry page0, size_t sk, size_t sv) {
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    const int bh = blockIdx.y, lo = blockIdx.x * TILE;
    auto pack = [](float a, float b) { return DT == 0 ? pk_h2(a, b) : pk_bf2(a, b); };
    if (dst_pt != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) {
        for (int p = threadIdx.x; p < pages; p += 256) {
            PageEntry e;
            e.k = page0.k + (size_t)p * sk;
            e.v = page0.v + (size_t)p * sv;
            dst_pt[p] = e;
        }
    }
    const PageEntry de = dst_pt != nullptr ? PageEntry{page0.k + (size_t)(lo >> PAGE_SHIFT) * sk, nullptr, page0.v + (size_t)(lo >> PAGE_SHIFT) * sv, nullptr}
                                           : dst.pt[lo >> PAGE_SHIFT];
    if (blockIdx.z == 0) {
        char *kdst = de.k + (size_t)bh * dst.k_cell + kfp_off(dst, lo, 0);
        const int upr = q.Dk / 32;  // units per row
        const uint32_t *krows = reinterpret_cast<const uint32_t *>(k_row_ptr(q, bh, lo));  // the tile's 64 rows are contiguous
        for (int u = threadIdx.x; u < upr * TILE; u += 256) {
            const int t = u / upr, p = u - t * upr;
            uint32_t w[BITS];
#pragma unroll
            for (int e = 0; e < BITS; ++e) w[e] = krows[(size_t)u * BITS + e];
            float sc, bi;
            pair_of<DT>(reinterpret_cast<const uint32_t *>(ksb_row_ptr(q, bh, lo + t))[(32 * p) / q.gs], sc, bi);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t o[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float x0 = __fadd_rn(__fmul_rn(sc, (float)unit_code<BITS, BITS>(w, (8 * k + 2 * j) * BITS)), bi);
                    const float x1 = __fadd_rn(__fmul_rn(sc, (float)unit_code<BITS, BITS>(w, (8 * k + 2 * j + 1) * BITS)), bi);
                    o[j] = pack(x0, x1);
                }
                *reinterpret_cast<u4v *>(kdst + ((size_t)(4 * p + k) * TILE + t) * 16) = u4v{o[0], o[1], o[2], o[3]};
            }
        }
        return;
    }
    // V: the pairs of the tile's 64 tokens, [group][token], through LDS
    extern __shared__ uint32_t sbv[];
    const int G = q.Dv / q.gs;
    for (int i = threadIdx.x; i < G * TILE; i += 256) {
        const int t = i / G, g = i - t * G;
        sbv[g * TILE + t] = reinterpret_cast<const uint32_t *>(vsb_row_ptr(q, bh, lo + t))[g];
    }
    __syncthreads();
    const uint32_t *vrows = reinterpret_cast<const uint32_t *>(v_cell_ptr(q, bh, lo) + v_row_off(q, lo, 0));  // Dv rows of 2 BITS dwords
    char *vdst = de.v + (size_t)bh * dst.v_cell + vfp_off(dst, lo, 0);
    for (int u = threadIdx.x; u < 2 * q.Dv; u += 256) {
        const int d = u >> 1, half = u & 1;
        uint32_t w[BITS];
#pragma unroll
        for (int e = 0; e < BITS; ++e) w[e] = vrows[(size_t)u * BITS + e];
        const uint32_t *sb = sbv + (d / q.gs) * TILE + 32 * half;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float s0, b0, s1, b1;
                pair_of<DT>(sb[8 * k + 2 * j], s0, b0);
                pair_of<DT>(sb[8 * k + 2 * j + 1], s1, b1);
                const float x0 = __fadd_rn(__fmul_rn(s0, (float)unit_code<BITS, BITS>(w, v_bitpos<BITS>(8 * k + 2 * j))), b0);
                const float x1 = __fadd_rn(__fmul_rn(s1, (float)unit_code<BITS, BITS>(w, v_bitpos<BITS>(8 * k + 2 * j + 1))), b1);
                o[j] = pack(x0, x1);
            }
            *reinterpret_cast<u4v *>(vdst + ((size_t)(4 * half + k) * q.Dv + d) * 16) = u4v{o[0], o[1], o[2], o[3]};
        }
    }
}

// grid (tiles touched x pieces of a tile, BH), 256 threads: rows src0 .. src0 + n - 1 to slots slot0 .. slot0 + n - 1, which
// may start and end inside a tile; ES bytes an element, keys of DK and values of DV.  A tile's K rows go in pieces of 4 to 32
// tokens, a 16-byte chunk to a thread, its V rows in blocks of columns that are turned through LDS: many short workgroups,
// whose loads are all in flight at once and whose threads form the sines of one chunk.  (A workgroup to a tile, as it was,
// walked four to sixteen chunks a thread: 512 rows of 8 heads x 128 with the queries of 32, 11.3 us.)
// HBM-bound from a few thousand rows on: 2048 rows of 64 (batch, head) pairs x 128, 16-bit 20.8 us, float32 40.1 (6.7
// TB/s); a row to a workgroup, whose values leave an element at a time, takes 113 us for the float32 rows, 70 for the
// 14.4 of 2048 rows of 64 pairs x 80 and 88 for the 22.4 of 2048 rows of 16 pairs x 512.
template <int ES, int DK, int DV> struct FpTile {
    static constexpr int E = 16 / ES;     // elements of a chunk
    static constexpr int TPRK = DK / E;   // chunks of a K row
    static constexpr int KT = TPRK <= 8 ? 32 : TPRK <= 16 ? 16 : TPRK <= 32 ? 8 : 4;        // tokens of a K piece
    static constexpr int KP = TILE / KT;
    static constexpr int VC = ES == 4 ? 32 : DV % 64 == 0 ? 64 : DV;                        // columns of a V piece
    static constexpr int VP = DV / VC;
    static constexpr int PIECES = KP + VP;
};
// the chunk `k` of `row` at d0, rotated
template <int DT>
__device__ __forceinline__ kv_u4 turned_chunk(const kv_u4 &k, const char *row, int d0, const RopeDev &rope, const float *inv_s, int pos) {
    float w[rope_chunk_elems<DT>()];
    if (rope.vec) {
        rope_chunk<DT>(rope, inv_s, row, d0, pos, k, w);
    } else {
#pragma unroll
        for (int j = 0; j < rope_chunk_elems<DT>(); ++j) w[j] = rope_elem<DT, true>(rope, row, d0 + j, pos);
    }
    return chunk_pack<DT>(w);
}
template <int ES, int DK, int DV>
__global__ void __launch_bounds__(256)
append_fp_tile_kernel(Store st, const char *keys, const char *values, int L, int src0, int slot0, int n, RopeDev rope) {
    using P = FpTile<ES, DK, DV>;
    using T = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
    constexpr int E = P::E, TPRK = P::TPRK, TPR = P::VC / E;  // chunks of a row, K and V (of the piece's columns)
    constexpr int VPW = P::VC * ES / 4 + 1;  // dword pitch of a token's V row in LDS (odd: column reads spread over banks)
    static_assert(DK % E == 0 && DV % P::VC == 0 && P::VC % E == 0 && P::KT * TPRK <= 256, "whole chunks, one to a thread");
    __shared__ uint32_t vt[TILE * VPW];
    __shared__ float inv_s[DK / 2];
    const int bh = blockIdx.y;
    if (bh >= st.BH) {  // queries of the same forward
        if constexpr (ES == 4) rope_queries_ride<2>(rope, st.BH, inv_s);
        else if (st.dtype == KVHIP_F16) rope_queries_ride<0>(rope, st.BH, inv_s);
        else rope_queries_ride<1>(rope, st.BH, inv_s);
        return;
    }
    const int piece = blockIdx.x % P::PIECES;
    const int slot_t = (slot0 & ~(TILE - 1)) + blockIdx.x / P::PIECES * TILE;
    const int l_t = src0 + slot_t - slot0;  // the row in the tile's first slot (before the first new row: t_lo > 0)
    // tokens [t_lo, t_hi) of the tile are new; the threads of the others repeat the nearest new row and write nothing
    const int t_lo = max(slot0 - slot_t, 0), t_hi = min(slot0 + n - slot_t, TILE);
    auto new_row = [&](int r) { return min(max(r, t_lo), t_hi - 1); };
    if (piece < P::KP) {
        if (piece * P::KT >= t_hi || (piece + 1) * P::KT <= t_lo) return;  // (workgroup-uniform)
        const int r = piece * P::KT + threadIdx.x / TPRK, d0 = (threadIdx.x % TPRK) * E, rn = new_row(r);
        const bool live = threadIdx.x < P::KT * TPRK;
        const char *row = keys + ((ptrdiff_t)bh * L + l_t + rn) * DK * ES;
        kv_u4 k{0u, 0u, 0u, 0u};
        if (live) k = *reinterpret_cast<const kv_u4 *>(row + ES * d0);
        if (rope.dims > 0) {
            rope_inv_table(rope, inv_s);
            __syncthreads();
            if (live && d0 < rope.dims) {
                const int pos = rope_pos(rope, bh, l_t + rn);
                if constexpr (ES == 4) k = turned_chunk<2>(k, row, d0, rope, inv_s, pos);
                else if (st.dtype == KVHIP_F16) k = turned_chunk<0>(k, row, d0, rope, inv_s, pos);
                else k = turned_chunk<1>(k, row, d0, rope, inv_s, pos);
            }
        }
        char *kcell = page_table(st)[slot_t >> PAGE_SHIFT].k + (size_t)bh * st.k_cell;  // a tile lies inside one page
        if (live && r >= t_lo && r < t_hi) *reinterpret_cast<kv_u4 *>(kcell + kfp_at<ES>(DK * ES, slot_t, 0) + kfp_at<ES>(DK * ES, r, d0)) = k;
        return;
    }
    const int c0 = (piece - P::KP) * P::VC;  // first column
    const char *vbase = values + (((ptrdiff_t)bh * L + l_t) * DV + c0) * ES;
    constexpr int CHUNKS = TILE * TPR, NV = (CHUNKS + 255) / 256;  // chunks of the piece, of a thread
    kv_u4 vraw[NV];
#pragma unroll
    for (int e = 0; e < NV; ++e) {
        const int c = min(e * 256 + (int)threadIdx.x, CHUNKS - 1), r = c / TPR;
        vraw[e] = *reinterpret_cast<const kv_u4 *>(vbase + (ptrdiff_t)new_row(r) * DV * ES + (c - r * TPR) * 16);
    }
#pragma unroll
    for (int e = 0; e < NV; ++e) {
        const int c = e * 256 + threadIdx.x, r = c / TPR;
        if (CHUNKS % 256 != 0 && c >= CHUNKS) break;
        uint32_t *vrow = &vt[r * VPW + (c - r * TPR) * 4];
        vrow[0] = vraw[e].x;
        vrow[1] = vraw[e].y;
        vrow[2] = vraw[e].z;
        vrow[3] = vraw[e].w;
    }
    __syncthreads();
    // chunks of E tokens of every column: a thread gathers tokens E ce .. E ce + E - 1 of column d;
    // consecutive threads take consecutive columns, so a chunk row is written contiguously
    char *cell = const_cast<char *>(v_cell_ptr(st, bh, slot_t)) + vfp_at<ES>(DV, slot_t, 0);
    const T *vte = reinterpret_cast<const T *>(vt);
    constexpr int VPE = VPW * 4 / ES;
    for (int c = threadIdx.x; c < P::VC * (TILE / E); c += 256) {
        const int t0 = c / P::VC * E, d = c % P::VC;
        uint32_t out[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (ES == 4) out[j] = vte[(t0 + j) * VPE + d];
            else out[j] = (uint32_t)vte[(t0 + 2 * j) * VPE + d] | ((uint32_t)vte[(t0 + 2 * j + 1) * VPE + d] << 16);
        }
        char *dst = cell + vfp_at<ES>(DV, t0, c0 + d);
        if (t0 >= t_lo && t0 + E <= t_hi) {
            *reinterpret_cast<kv_u4 *>(dst) = kv_u4{out[0], out[1], out[2], out[3]};
        } else {
#pragma unroll
            for (int j = 0; j < E; ++j)
                if (t0 + j >= t_lo && t0 + j < t_hi) reinterpret_cast<T *>(dst)[j] = (T)(ES == 4 ? out[j] : out[j / 2] >> (16 * (j & 1)));
        }
    }
}

template <int ES>
__global__ void export_fp_kernel(Store st, Runs runs, int row_begin, int dst_row0, int nrows, char *dst_k, char *dst_v) {
    const int bh = blockIdx.y;
    const int slot = row_to_slot(runs, row_begin + blockIdx.x);
    const int i = row_begin + blockIdx.x - dst_row0;  // row of the dense destination [BH, nrows, D]
    if (slot < 0) return;
    using E = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
    if (dst_k) {
        const char *kc = k_cell_ptr(st, bh, slot);
        E *kd = reinterpret_cast<E *>(dst_k) + ((size_t)bh * nrows + i) * st.Dk;
        for (int d = threadIdx.x; d < st.Dk; d += blockDim.x) kd[d] = *reinterpret_cast<const E *>(kc + kfp_off(st, slot, d));
    }
    if (dst_v) {
        const char *vc = v_cell_ptr(st, bh, slot);
        E *vd = reinterpret_cast<E *>(dst_v) + ((size_t)bh * nrows + i) * st.Dv;
        for (int d = threadIdx.x; d < st.Dv; d += blockDim.x)
            vd[d] = *reinterpret_cast<const E *>(vc + vfp_off(st, slot, d));
    }
}

template <int ES>
__global__ void import_fp_kernel(Store st, const char *src_k, const char *src_v, int nrows) {
    const int bh = blockIdx.y;
    const int slot = blockIdx.x;
    using E = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
    const E *ks = reinterpret_cast<const E *>(src_k) + ((size_t)bh * nrows + slot) * st.Dk;
    char *kc = const_cast<char *>(k_cell_ptr(st, bh, slot));
    for (int d = threadIdx.x; d < st.Dk; d += blockDim.x) *reinterpret_cast<E *>(kc + kfp_off(st, slot, d)) = ks[d];
    const E *vs = reinterpret_cast<const E *>(src_v) + ((size_t)bh * nrows + slot) * st.Dv;
    char *vc = const_cast<char *>(v_cell_ptr(st, bh, slot));
    for (int d = threadIdx.x; d < st.Dv; d += blockDim.x) *reinterpret_cast<E *>(vc + vfp_off(st, slot, d)) = vs[d];
}

// Rows in presented order into slots 0, 1, ... of another store (a ring that is laid out again, a copy).  grid (chunks of
// 16 / ES rows, BH), 256 threads: the rows' 16-byte K chunks move whole, lanes along the rows; a thread puts a column's V
// chunk together from the two that hold its tokens, shifted by where the run starts.  Chunks that a run begins or ends
// inside (and rows of another launch's runs) go element by element.  A ring of 4096 rows of 16 (batch, head) pairs x 256,
// 16-bit (134 MB in and out): 34.7 us; 43 with offsets that divide by the element size, three divisions to a chunk and side;
// element by element 155 us.
template <int ES>
__global__ void __launch_bounds__(256) compact_fp_kernel(Store src, Runs runs, Store dst, int nrows) {
    using E = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
    constexpr int EPC = 16 / ES;
    const int bh = blockIdx.y, i0 = blockIdx.x * EPC, tid = threadIdx.x;
    int slot[EPC];
    bool run = true;  // (all of this is workgroup-uniform)
#pragma unroll
    for (int j = 0; j < EPC; ++j) {
        slot[j] = i0 + j < nrows ? row_to_slot(runs, i0 + j) : -1;
        run = run && slot[j] >= 0 && slot[j] == slot[0] + j;
    }
    const int row = i0 + tid % EPC, from = row < nrows ? row_to_slot(runs, row) : -1;
    if (from >= 0) {
        const char *ks = k_cell_ptr(src, bh, from);
        char *kd = const_cast<char *>(k_cell_ptr(dst, bh, row));
        const int chunks = src.Dk / EPC;
        for (int c = tid / EPC; c < chunks; c += 256 / EPC)
            *reinterpret_cast<kv_u4 *>(kd + kfp_at<ES>(dst.k_row, row, c * EPC)) = *reinterpret_cast<const kv_u4 *>(ks + kfp_at<ES>(src.k_row, from, c * EPC));
        for (int d = chunks * EPC + tid / EPC; d < src.Dk; d += 256 / EPC)
            *reinterpret_cast<E *>(kd + kfp_at<ES>(dst.k_row, row, d)) = *reinterpret_cast<const E *>(ks + kfp_at<ES>(src.k_row, from, d));
    }
    if (run) {
        const int sh = slot[0] % EPC, last = slot[0] + EPC - 1;
        const char *v0 = v_cell_ptr(src, bh, slot[0]), *v1 = v_cell_ptr(src, bh, last);
        char *vd = const_cast<char *>(v_cell_ptr(dst, bh, i0));
        for (int d = tid; d < src.Dv; d += 256) {
            const kv_u4 x = *reinterpret_cast<const kv_u4 *>(v0 + vfp_at<ES>(src.Dv, slot[0] - sh, d));
            const kv_u4 y = *reinterpret_cast<const kv_u4 *>(v1 + vfp_at<ES>(src.Dv, last - last % EPC, d));
            uint32_t w[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
            const int words = sh * ES / 4;  // whole words to drop in front
            if (words & 2) {
#pragma unroll
                for (int k = 0; k < 6; ++k) w[k] = w[k + 2];
            }
            if (words & 1) {
#pragma unroll
                for (int k = 0; k < 5; ++k) w[k] = w[k + 1];
            }
            if (ES == 2 && (sh & 1)) {
#pragma unroll
                for (int k = 0; k < 4; ++k) w[k] = (w[k] >> 16) | (w[k + 1] << 16);
            }
            *reinterpret_cast<kv_u4 *>(vd + vfp_at<ES>(dst.Dv, i0, d)) = kv_u4{w[0], w[1], w[2], w[3]};
        }
        return;
    }
    for (int j = 0; j < EPC; ++j) {
        const int at = i0 + j < nrows ? row_to_slot(runs, i0 + j) : -1;
        if (at < 0) continue;
        const char *vs = v_cell_ptr(src, bh, at);
        char *vd = const_cast<char *>(v_cell_ptr(dst, bh, i0 + j));
        for (int d = tid; d < src.Dv; d += 256)
            *reinterpret_cast<E *>(vd + vfp_at<ES>(dst.Dv, i0 + j, d)) = *reinterpret_cast<const E *>(vs + vfp_at<ES>(src.Dv, at, d));
    }
}

// The arrays of a quantized state, any of the six (null: not asked for).  grid (64-token tiles, BH), 256 threads: K rows
// are contiguous in page and array alike and are copied (VEC: as 16-byte pieces); V rows are put together from the
// transposed tile, 128 columns at a time through LDS, lanes taking the tokens of a column (their codes lie in adjacent
// dwords: no bank conflicts); pairs are split into scales and biases.  A row to a workgroup and an array to a launch,
// as it was, takes 19 us an array for 5000 rows of 16 (batch, head) pairs x 128 at 4 bits; four such caches converted
// and read out: 630 us then, 188 us in one launch a cache.
template <int BITS, bool VEC>
__global__ void __launch_bounds__(256) export_quant_kernel(Store st, QuantArrays out, int nrows) {
    constexpr int CB = 128;  // columns per round
    __shared__ __attribute__((aligned(16))) uint32_t vs[CB * 2 * BITS];
    const int bh = blockIdx.y, lo = blockIdx.x * TILE, n = min(TILE, nrows - lo);
    const int tid = threadIdx.x;
    const size_t row0 = (size_t)bh * nrows + lo;
    if (out.a[0]) {
        const char *src = k_row_ptr(st, bh, lo);
        char *dst = static_cast<char *>(out.a[0]) + row0 * st.k_row;
        if (VEC) {
            for (int i = tid; i < n * (int)(st.k_row / 16); i += 256)
                reinterpret_cast<u4v *>(dst)[i] = reinterpret_cast<const u4v *>(src)[i];
        } else {
            for (int i = tid; i < n * (int)(st.k_row / 4); i += 256)
                reinterpret_cast<uint32_t *>(dst)[i] = reinterpret_cast<const uint32_t *>(src)[i];
        }
    }
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        void *sc = out.a[1 + 3 * side], *bi = out.a[2 + 3 * side];
        if (!sc && !bi) continue;
        const char *src = side == 0 ? ksb_row_ptr(st, bh, lo) : vsb_row_ptr(st, bh, lo);
        const int G = (side == 0 ? st.Dk : st.Dv) / st.gs;
        for (int i = tid; i < n * G; i += 256) {
            if (st.es == 2) {
                const uint32_t pair = reinterpret_cast<const uint32_t *>(src)[i];
                if (sc) reinterpret_cast<uint16_t *>(sc)[row0 * G + i] = (uint16_t)pair;
                if (bi) reinterpret_cast<uint16_t *>(bi)[row0 * G + i] = (uint16_t)(pair >> 16);
            } else {
                const uint2 pair = reinterpret_cast<const uint2 *>(src)[i];
                if (sc) reinterpret_cast<uint32_t *>(sc)[row0 * G + i] = pair.x;
                if (bi) reinterpret_cast<uint32_t *>(bi)[row0 * G + i] = pair.y;
            }
        }
    }
    if (!out.a[3]) return;
    const int W = st.Dv * BITS / 32;
    const char *cell = v_cell_ptr(st, bh, lo) + v_row_off(st, lo, 0);
    uint32_t *dst = static_cast<uint32_t *>(out.a[3]) + row0 * W;
    for (int c0 = 0; c0 < st.Dv; c0 += CB) {
        const int cols = min(CB, st.Dv - c0), words = cols * BITS / 32;  // (head sizes are multiples of 32 columns)
        __syncthreads();
        for (int i = tid; i < cols * BITS / 2; i += 256)
            reinterpret_cast<u4v *>(vs)[i] = reinterpret_cast<const u4v *>(cell + (size_t)c0 * (8 * BITS))[i];
        __syncthreads();
        auto word_of = [&](int t, int w) -> uint32_t {
            uint32_t word = 0;
            if constexpr ((32 % BITS) == 0) {
                constexpr int per = 32 / BITS;
#pragma unroll
                for (int i = 0; i < per; ++i)
                    word |= v_code_load<BITS>(reinterpret_cast<const char *>(vs + (w * per + i) * 2 * BITS), t) << (i * BITS);
            } else {
                const int j0 = (32 * w) / BITS;  // the first column with bits in word w of the row's bit stream
#pragma unroll
                for (int i = 0; i < 32 / BITS + 2; ++i) {
                    const int j = j0 + i;
                    if (j < cols && j * BITS < 32 * w + 32)
                        word |= stream_bits(v_code_load<BITS>(reinterpret_cast<const char *>(vs + j * 2 * BITS), t), j * BITS, w);
                }
            }
            return word;
        };
        const int t = tid & (TILE - 1);
        if (t >= n) continue;
        uint32_t *row = dst + (size_t)t * W + c0 * BITS / 32;
        if (VEC && words % 4 == 0) {
            for (int w = (tid >> 6) * 4; w < words; w += 16)
                *reinterpret_cast<u4v *>(row + w) = u4v{word_of(t, w), word_of(t, w + 1), word_of(t, w + 2), word_of(t, w + 3)};
        } else {
            for (int w = tid >> 6; w < words; w += 4) row[w] = word_of(t, w);
        }
    }
}

// grid (64-token tiles, BH): dense reference arrays into slots [0, nrows)
template <int BITS>
__global__ void import_quant_kernel(Store st, const uint32_t *kw, const char *ks, const char *kb,
                                    const uint32_t *vw, const char *vs, const char *vb, int nrows) {
    const int bh = blockIdx.y;
    const int lo = blockIdx.x * TILE, hi = min(nrows, lo + TILE);
    const int es = st.es;
    const int Wk = st.Dk * BITS / 32, Wv = st.Dv * BITS / 32, Gk = st.Dk / st.gs, Gv = st.Dv / st.gs;
    for (int slot = lo; slot < hi; ++slot) {
        const size_t r = (size_t)bh * nrows + slot;
        uint32_t *kd = reinterpret_cast<uint32_t *>(const_cast<char *>(k_row_ptr(st, bh, slot)));
        for (int w = threadIdx.x; w < Wk; w += blockDim.x) kd[w] = kw[r * Wk + w];
        char *ksd = const_cast<char *>(ksb_row_ptr(st, bh, slot));
        char *vsd = const_cast<char *>(vsb_row_ptr(st, bh, slot));
        for (int g = threadIdx.x; g < Gk; g += blockDim.x) {
            if (es == 2) {
                reinterpret_cast<uint16_t *>(ksd)[2 * g] = reinterpret_cast<const uint16_t *>(ks)[r * Gk + g];
                reinterpret_cast<uint16_t *>(ksd)[2 * g + 1] = reinterpret_cast<const uint16_t *>(kb)[r * Gk + g];
            } else {
                reinterpret_cast<uint32_t *>(ksd)[2 * g] = reinterpret_cast<const uint32_t *>(ks)[r * Gk + g];
                reinterpret_cast<uint32_t *>(ksd)[2 * g + 1] = reinterpret_cast<const uint32_t *>(kb)[r * Gk + g];
            }
        }
        for (int g = threadIdx.x; g < Gv; g += blockDim.x) {
            if (es == 2) {
                reinterpret_cast<uint16_t *>(vsd)[2 * g] = reinterpret_cast<const uint16_t *>(vs)[r * Gv + g];
                reinterpret_cast<uint16_t *>(vsd)[2 * g + 1] = reinterpret_cast<const uint16_t *>(vb)[r * Gv + g];
            } else {
                reinterpret_cast<uint32_t *>(vsd)[2 * g] = reinterpret_cast<const uint32_t *>(vs)[r * Gv + g];
                reinterpret_cast<uint32_t *>(vsd)[2 * g + 1] = reinterpret_cast<const uint32_t *>(vb)[r * Gv + g];
            }
        }
    }
    char *cell = const_cast<char *>(v_cell_ptr(st, bh, lo));
    constexpr int TPW = 32 / BITS;
    constexpr int WPR = TILE * BITS / 32;
    for (int u = threadIdx.x; u < st.Dv * WPR; u += blockDim.x) {
        const int d = u / WPR, w = u - d * WPR;
        uint32_t nbits = 0;
        if constexpr ((32 % BITS) == 0) {
            for (int tt = 0; tt < TPW; ++tt) {
                const int t = w * TPW + tt;
                if (lo + t < hi)
                    nbits |= stream_code<BITS>(vw + ((size_t)bh * nrows + lo + t) * Wv, d) << (v_bitpos<BITS>(t) & 31);
            }
        } else {
            const int t0 = (32 * w) / BITS;  // the first token with bits in word w of the tile row
            for (int tt = 0; tt < TPW + 2; ++tt) {
                const int t = t0 + tt;
                if (t < TILE && lo + t < hi && t * BITS < 32 * w + 32)
                    nbits |= stream_bits(stream_code<BITS>(vw + ((size_t)bh * nrows + lo + t) * Wv, d), t * BITS, w);
            }
        }
        reinterpret_cast<uint32_t *>(cell + v_row_off(st, lo, d))[w] = nbits;
    }
}

// one wavefront per row; grid.x * 4 waves
template <int DT, int BITS>
__global__ void __launch_bounds__(256)
affine_quantize_kernel(const char *src, int64_t rows, int D, int gs, uint32_t *wq, char *scales, char *biases, int es) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int W = D * BITS / 32, G = D / gs;
    quantize_row_wave<DT, BITS>(src + row * D * es, D, gs, lane, wq + row * W, nullptr, nullptr,
                                scales + row * G * es, biases + row * G * es);
}

template <int DT, int BITS>
__global__ void affine_dequantize_kernel(const uint32_t *wq, const char *scales, const char *biases,
                                         int64_t rows, int D, int gs, char *dst) {
    const int64_t row = blockIdx.x;
    const int W = D * BITS / 32, G = D / gs;
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        const uint32_t c = stream_code<BITS>(wq + row * W, d);
        const float s = Elem<DT>::load(scales, row * G + d / gs);
        const float b = Elem<DT>::load(biases, row * G + d / gs);
        Elem<DT>::store(dst, row * D + d, __fadd_rn(__fmul_rn(s, (float)c), b));
    }
}

__global__ void mask_materialize_kernel(kvhip_mask_plan_t p, uint8_t *dst) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= p.cols) return;
    if (p.rolled) {
        // (arange(cols) >= cols - window) rolled right by roll_shift
        const int src = ((j - p.roll_shift) % p.cols + p.cols) % p.cols;
        dst[j] = src >= p.cols - p.roll_window;
        return;
    }
    for (int i = blockIdx.y; i < p.rows; i += gridDim.y) {
        const int li = p.offset + i;
        bool keep = li >= j;
        if (p.window > 0) keep = keep && (li < j + p.window);
        dst[(size_t)i * p.cols + j] = keep;
    }
}

}  // namespace

#define KV_DISPATCH_DT_BITS(DTV, BITSV, CALL)                                                  \
    do {                                                                                       \
        if ((BITSV) == 4) { if ((DTV) == 0) { CALL(0, 4); } else if ((DTV) == 1) { CALL(1, 4); } else { CALL(2, 4); } } \
        else if ((BITSV) == 8) { if ((DTV) == 0) { CALL(0, 8); } else if ((DTV) == 1) { CALL(1, 8); } else { CALL(2, 8); } } \
        else if ((BITSV) == 3) { if ((DTV) == 0) { CALL(0, 3); } else if ((DTV) == 1) { CALL(1, 3); } else { CALL(2, 3); } } \
        else if ((BITSV) == 5) { if ((DTV) == 0) { CALL(0, 5); } else if ((DTV) == 1) { CALL(1, 5); } else { CALL(2, 5); } } \
        else if ((BITSV) == 6) { if ((DTV) == 0) { CALL(0, 6); } else if ((DTV) == 1) { CALL(1, 6); } else { CALL(2, 6); } } \
        else { if ((DTV) == 0) { CALL(0, 2); } else if ((DTV) == 1) { CALL(1, 2); } else { CALL(2, 2); } } \
    } while (0)

namespace {
thread_local int g_last_append = -1;
// The caller's rotation as this launch takes it: queries that ride along ride once.
RopeDev take_rope(RopeDev *rope) {
    if (!rope) return RopeDev();
    const RopeDev r = *rope;
    rope->qx = nullptr;
    return r;
}

hipError_t launch_append_fp_rows(const Store &st, const void *keys, const void *values, int L, int src0,
                                 int slot0, int n, hipStream_t s, const RopeDev &r) {
    if (n <= 0) return hipSuccess;
    g_last_append = 0;
    const dim3 block(r.qx ? 256 : 128), grid(n, st.BH + rope_ride_rows(r, n, st.es, block.x));
    // (without queries an instance of its own: their LDS table cost the plain append of 512 rows of 64 (batch, head) pairs x 80
    // 25 us instead of 21)
#define FP_ROWS(ES, RIDE) hipLaunchKernelGGL((append_fp_kernel<ES, RIDE>), grid, block, 0, s, st, (const char *)keys, (const char *)values, L, src0, slot0, r)
    if (st.es == 2) {
        if (r.qx) FP_ROWS(2, true);
        else FP_ROWS(2, false);
    } else {
        if (r.qx) FP_ROWS(4, true);
        else FP_ROWS(4, false);
    }
#undef FP_ROWS
    return hipGetLastError();
}
}  // namespace

int last_append_kernel() { return g_last_append; }

hipError_t launch_append_fp(const Store &st, const void *keys, const void *values, int L, int src0,
                            int slot0, int n, hipStream_t s, RopeDev *rope) {
    if (n <= 0) return hipSuccess;
    const RopeDev r = take_rope(rope);
    // One launch for whole tiles and the pieces of tiles at either end.  Few rows go one to a workgroup, which takes 3 us
    // until there are more of them than run at once.  Row / tile kernel, us: 16-bit rows x 128, of 128 (batch, head) pairs,
    // 8 each 3.1 / 3.5, 16 4.3 / 3.5, 63 9.0 / 4.0; of 8 pairs, 63 each 2.8 / 3.1; x 256, 32 pairs, 16 each 3.5 / 3.5, 24
    // 3.8 / 3.4; x 64, 128 pairs, 16 each 3.3 / 3.2, 32 4.6 / 3.2; float32 x 128, 32 pairs, 16 each 3.1 / 3.0, 48 4.3 / 3.1.
    // (Queries that ride are the longer part of whichever launch takes them.)
    const bool many = n >= 16 && (size_t)n * st.BH * (st.Dk + st.Dv) * st.es > (512u << 10);
    if (!many && (n < TILE || !r.qx)) return launch_append_fp_rows(st, keys, values, L, src0, slot0, n, s, r);
    const int tiles = ((slot0 & (TILE - 1)) + n + TILE - 1) / TILE;
#define FP_TILE(ES, DK, DV)                                                                                               \
    do {                                                                                                                  \
        const int gx = tiles * FpTile<ES, DK, DV>::PIECES;                                                                \
        g_last_append = 1;                                                                                                \
        hipLaunchKernelGGL((append_fp_tile_kernel<ES, DK, DV>), dim3(gx, st.BH + rope_ride_rows(r, gx, st.es, 256)), dim3(256), 0, s, st, \
                           (const char *)keys, (const char *)values, L, src0, slot0, n, r);                               \
        return hipGetLastError();                                                                                         \
    } while (0)
    if (st.es == 2) {
        if (st.Dk == 192 && st.Dv == 128) FP_TILE(2, 192, 128);
        if (st.Dk == st.Dv) {
            if (st.Dk == 64) FP_TILE(2, 64, 64);
            if (st.Dk == 80) FP_TILE(2, 80, 80);
            if (st.Dk == 96) FP_TILE(2, 96, 96);
            if (st.Dk == 128) FP_TILE(2, 128, 128);
            if (st.Dk == 256) FP_TILE(2, 256, 256);
            if (st.Dk == 512) FP_TILE(2, 512, 512);
        }
    } else if (st.Dk == st.Dv) {
        if (st.Dk == 64) FP_TILE(4, 64, 64);
        if (st.Dk == 96) FP_TILE(4, 96, 96);
        if (st.Dk == 128) FP_TILE(4, 128, 128);
        if (st.Dk == 256) FP_TILE(4, 256, 256);
    }
#undef FP_TILE
    return launch_append_fp_rows(st, keys, values, L, src0, slot0, n, s, r);  // other head sizes
}

hipError_t launch_rope_apply(const RopeDev &rope, const void *x, void *out, int B, int H, int L, int D,
                             int dtype, hipStream_t s) {
    if ((size_t)B * H * L == 0) return hipSuccess;
    if (rope.vec) {
        const int hg = rope_heads_per_group(L * B, H, D, dtype == KVHIP_F32 ? 4 : 2, 256);
#define ROPE_ROWS(DT) hipLaunchKernelGGL(rope_rows_kernel<DT>, dim3(L, B, (H + hg - 1) / hg), dim3(256), 0, s, rope, (const char *)x, (char *)out, H, L, D)
        if (dtype == KVHIP_F16) ROPE_ROWS(0);
        else if (dtype == KVHIP_BF16) ROPE_ROWS(1);
        else ROPE_ROWS(2);
#undef ROPE_ROWS
        return hipGetLastError();
    }
    dim3 grid(L, B * H), block(D <= 64 ? 64 : (D <= 128 ? 128 : 256));  // at most 4 elements per thread up to D = 1024
    if (dtype == KVHIP_F16) hipLaunchKernelGGL(rope_apply_kernel<0>, grid, block, 0, s, rope, (const char *)x, (char *)out, L, D);
    else if (dtype == KVHIP_BF16) hipLaunchKernelGGL(rope_apply_kernel<1>, grid, block, 0, s, rope, (const char *)x, (char *)out, L, D);
    else hipLaunchKernelGGL(rope_apply_kernel<2>, grid, block, 0, s, rope, (const char *)x, (char *)out, L, D);
    return hipGetLastError();
}

namespace {
hipError_t launch_append_quant_rows(const Store &st, const void *keys, const void *values, int L, int src0,
                                    int slot0, int n, hipStream_t s, const RopeDev &r) {
    if (n <= 0) return hipSuccess;
    g_last_append = 0;
    const int ntile = ((slot0 + n - 1) >> 6) - (slot0 >> 6) + 1;
    // (a speculative-verify step appends 4 rows: 8 (row, K or V) items, one per wavefront)
    const dim3 block(n >= 3 ? 512 : 256), grid(ntile, st.BH + rope_ride_rows(r, ntile, st.es, block.x));
    const size_t lds = (size_t)TILE * st.Dv;
#define CALL(DT, BITS)                                                                                      \
    do {                                                                                                    \
        if (r.dims > 0)                                                                                     \
            hipLaunchKernelGGL((append_quant_kernel<DT, BITS, true>), grid, block, lds, s, st, (const char *)keys,  \
                               (const char *)values, L, src0, slot0, n, r);                                 \
        else                                                                                                \
            hipLaunchKernelGGL((append_quant_kernel<DT, BITS, false>), grid, block, lds, s, st, (const char *)keys, \
                               (const char *)values, L, src0, slot0, n, r);                                 \
    } while (0)
    KV_DISPATCH_DT_BITS(st.dtype, st.bits, CALL);
#undef CALL
    return hipGetLastError();
}
}  // namespace

// Rows in one tile from which the tile quantizer is the faster one.  The row kernel's wavefronts take their rows one
// after the other, 64 columns at a time (128 with groups of 128); a tile takes its time whatever its rows.  Row / tile
// kernel, us, 4 bits, 128 (batch, head) pairs: x 128 rotated 5.5 / 5.2 for 2 rows, 6.0 / 5.3 for 4, 11.2 / 5.6 for 11;
// as they are 4.6 / 5.0 for 4, 5.8 / 5.2 for 5; x 256, groups of 128, 7.4 / 5.9 rotated for 3 and 5.5 / 6.0, 7.1 / 6.0 for
// 4 and 5; x 64 5.0 / 4.8 rotated for 4, 4.0 / 4.0 and 4.7 / 4.0 for 4 and 6.  Keys of 192 with values of 128 take two
// launches: 9.4 / 9.6 for 9 and 10.8 / 9.6 for 12, rotated 13.6 / 12.6 and 15.2 / 12.3.
// Where the tile kernel's pieces no longer run at once and the row kernel's workgroups still do, the line lies higher.  Tile
// less row kernel, us, 256 and 512 pairs: rotated, 4 rows, 4 bits x 128 +0.1 and +0.8, 8 bits +0.8 and +1.0 (128 pairs -0.6,
// -0.2; 1024 pairs -1.0, -0.9), 5 rows -1.7 and -1.8, -1.2 and -1.3, but 3 bits -1.4 and -2.4 for 4; as they are, 5 rows, 4
// bits +0.2 and +0.8, 8 bits +1.6 and +0.9, x 64 +0.3 and +0.5, 3 bits -0.6 and -0.4, 6 bits x 64 +0.4 and +0.6; x 256 in
// groups of 128 +0.1 and +1.9 for 8 rows, -3.4 and -2.4 for 12; keys of 192 rotated, 512 pairs, +0.9 for 12, -5.0 for 16.
int quant_tile_rows(const Store &st, bool rotated) {
    const bool between = st.BH > 128 && st.BH < 1024, stream = st.bits != 4 && st.bits != 8;
    if (quant_tiles_two_sided(st)) return rotated && between && st.BH > 256 ? 14 : 12;
    if (rotated) return between && !stream ? 5 : 3;
    if (!between || (stream && st.Dk > 64)) return 5;
    return st.Dk == 256 && st.gs == 128 ? 12 : 8;
}

hipError_t launch_append_quant(const Store &st, const void *keys, const void *values, int L, int src0,
                               int slot0, int n, hipStream_t s, RopeDev *rope) {
    if (n <= 0) return hipSuccess;
    const RopeDev r = take_rope(rope);
    const bool tiled = quant_tiles_one_launch(st) || quant_tiles_two_sided(st);
    // One launch of the tile kernel takes every row of its tiles at once, 4 to 12 us whatever their number; the row kernel's
    // wavefronts take theirs one after the other, each tile's in a workgroup of its own (33 us for 50 rows of 128).
    // A 501-row piece at an odd slot, rotated: 50 us as rows, whole tiles, rows (three launches), 7 us so.
    const int head = std::min(n, TILE - (slot0 & (TILE - 1)));
    const int most = std::max(head, std::min(n - head, TILE));
    if (!tiled || most < quant_tile_rows(st, r.dims > 0)) return launch_append_quant_rows(st, keys, values, L, src0, slot0, n, s, r);
    g_last_append = 1;
    if (st.bits == 4) return launch_quant_tiles_bits<4, true, false>(st, st, keys, values, L, src0, slot0, n, s, r);
    if (st.bits == 8) return launch_quant_tiles_bits<8, true, false>(st, st, keys, values, L, src0, slot0, n, s, r);
    return launch_quant_tiles_other(st, keys, values, L, src0, slot0, n, s, r);
}

hipError_t launch_requant_pages(const Store &src, const Store &st, int rows, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const int tiles = (rows + TILE - 1) / TILE;
    if (!quant_tiles_one_launch(st) && !quant_tiles_two_sided(st)) {
        dim3 grid(tiles, st.BH), block(256);
        const size_t lds = (size_t)TILE * st.Dv;
#define CALL(DT, BITS) hipLaunchKernelGGL((requant_rows_kernel<DT, BITS>), grid, block, lds, s, st, src, 0, rows)
        KV_DISPATCH_DT_BITS(st.dtype, st.bits, CALL);
#undef CALL
        return hipGetLastError();
    }
    // whole tiles, the last one included: its rows past `rows` hold zeros or rows trimmed earlier, and
    // what they quantize to lies past the new cache's offset, where the next append overwrites it
    const RopeDev none;
    if (st.bits == 4) return launch_quant_tiles_bits<4, true, true>(st, src, nullptr, nullptr, 0, 0, 0, rows, s, none);
    if (st.bits == 8) return launch_quant_tiles_bits<8, true, true>(st, src, nullptr, nullptr, 0, 0, 0, rows, s, none);
    return launch_requant_tiles_other(src, st, rows, s);
}

hipError_t launch_dequant_pages(const Store &q, const Store &dst, int rows, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    dim3 grid((rows + TILE - 1) / TILE, q.BH), block(256);
    if (q.es == 2 && q.Dk % 8 == 0 && q.Dv % 8 == 0) {
        const size_t lds = (size_t)(q.Dv / q.gs) * TILE * 4;
#define CALL(DT, BITS)                                                                                                  \
    do {                                                                                                                \
        if (q.Dk % 32 == 0 && q.Dv % 32 == 0)                                                                           \
            hipLaunchKernelGGL((dequant_units_kernel<(DT == 2 ? 0 : DT), BITS>), dim3(grid.x, grid.y, 2), block, lds, s, q, dst, \
                               (PageEntry *)nullptr, 0, PageEntry(), (size_t)0, (size_t)0);                             \
        else                                                                                                            \
            hipLaunchKernelGGL((dequant_tiles16_kernel<(DT == 2 ? 0 : DT), BITS>), dim3(grid.x, grid.y, 2), block, 0, s, q, dst, \
                               (PageEntry *)nullptr, 0, PageEntry(), (size_t)0, (size_t)0);                             \
    } while (0)
        KV_DISPATCH_DT_BITS(q.dtype, q.bits, CALL);
#undef CALL
        return hipGetLastError();
    }
#define CALL(DT, BITS) hipLaunchKernelGGL((dequant_pages_kernel<DT, BITS>), grid, block, 0, s, q, dst, rows)
    KV_DISPATCH_DT_BITS(q.dtype, q.bits, CALL);
#undef CALL
    return hipGetLastError();
}

// The same into scratch pages whose table the launch writes itself (16-bit dtypes, head sizes that are multiples of 8):
// page p of the scratch at `page0` + p * (sk, sv), `dst.pt` the table to fill, `dst` otherwise only geometry.
hipError_t launch_dequant_scratch(const Store &q, const Store &dst, int rows, int pages, const PageEntry &page0, size_t sk, size_t sv,
                                  hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (q.es != 2 || q.Dk % 8 != 0 || q.Dv % 8 != 0) return hipErrorInvalidValue;
    dim3 grid((rows + TILE - 1) / TILE, q.BH, 2), block(256);
    const size_t lds = (size_t)(q.Dv / q.gs) * TILE * 4;
#define CALL(DT, BITS)                                                                                          \
    do {                                                                                                        \
        if (q.Dk % 32 == 0 && q.Dv % 32 == 0)                                                                   \
            hipLaunchKernelGGL((dequant_units_kernel<(DT == 2 ? 0 : DT), BITS>), grid, block, lds, s, q, dst,    \
                               const_cast<PageEntry *>(dst.pt), pages, page0, sk, sv);                          \
        else                                                                                                    \
            hipLaunchKernelGGL((dequant_tiles16_kernel<(DT == 2 ? 0 : DT), BITS>), grid, block, 0, s, q, dst,    \
                               const_cast<PageEntry *>(dst.pt), pages, page0, sk, sv);                          \
    } while (0)
    KV_DISPATCH_DT_BITS(q.dtype, q.bits, CALL);
#undef CALL
    return hipGetLastError();
}

hipError_t launch_export_fp(const Store &st, const Runs &runs, int row_begin, int count, int dst_row0,
                            int dst_rows, void *dst_k, void *dst_v, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    dim3 grid(count, st.BH), block(128);
    if (st.es == 2)
        hipLaunchKernelGGL(export_fp_kernel<2>, grid, block, 0, s, st, runs, row_begin, dst_row0, dst_rows, (char *)dst_k, (char *)dst_v);
    else
        hipLaunchKernelGGL(export_fp_kernel<4>, grid, block, 0, s, st, runs, row_begin, dst_row0, dst_rows, (char *)dst_k, (char *)dst_v);
    return hipGetLastError();
}

hipError_t launch_import_fp(const Store &st, const void *src_k, const void *src_v, int nrows, hipStream_t s) {
    if (nrows <= 0) return hipSuccess;
    dim3 grid(nrows, st.BH), block(128);
    if (st.es == 2)
        hipLaunchKernelGGL(import_fp_kernel<2>, grid, block, 0, s, st, (const char *)src_k, (const char *)src_v, nrows);
    else
        hipLaunchKernelGGL(import_fp_kernel<4>, grid, block, 0, s, st, (const char *)src_k, (const char *)src_v, nrows);
    return hipGetLastError();
}

hipError_t launch_compact_fp(const Store &src, const Runs &runs, const Store &dst, int nrows, hipStream_t s) {
    if (nrows <= 0) return hipSuccess;
    const int per_wg = 16 / src.es;
    dim3 grid((nrows + per_wg - 1) / per_wg, src.BH), block(256);
    if (src.es == 2)
        hipLaunchKernelGGL(compact_fp_kernel<2>, grid, block, 0, s, src, runs, dst, nrows);
    else
        hipLaunchKernelGGL(compact_fp_kernel<4>, grid, block, 0, s, src, runs, dst, nrows);
    return hipGetLastError();
}

hipError_t launch_export_quant(const Store &st, const QuantArrays &out, int nrows, hipStream_t s) {
    if (nrows <= 0) return hipSuccess;
    dim3 grid((nrows + TILE - 1) / TILE, st.BH), block(256);
    // 16-byte pieces where every row of both code arrays starts on a 16-byte boundary
    const bool vec = st.k_row % 16 == 0 && (st.Dv * st.bits / 8) % 16 == 0 &&
                     ((reinterpret_cast<uintptr_t>(out.a[0]) | reinterpret_cast<uintptr_t>(out.a[3])) & 15) == 0;
#define EXP(BITS)                                                                                        \
    do {                                                                                                 \
        if (vec) hipLaunchKernelGGL((export_quant_kernel<BITS, true>), grid, block, 0, s, st, out, nrows); \
        else hipLaunchKernelGGL((export_quant_kernel<BITS, false>), grid, block, 0, s, st, out, nrows);    \
    } while (0)
    switch (st.bits) {
        case 4: EXP(4); break;
        case 8: EXP(8); break;
        case 3: EXP(3); break;
        case 5: EXP(5); break;
        case 6: EXP(6); break;
        default: EXP(2); break;
    }
#undef EXP
    return hipGetLastError();
}

hipError_t launch_import_quant(const Store &st, const void *const srcs[6], int nrows, hipStream_t s) {
    if (nrows <= 0) return hipSuccess;
    dim3 grid((nrows + TILE - 1) / TILE, st.BH), block(256);
#define IMP(BITS)                                                                                     \
    hipLaunchKernelGGL(import_quant_kernel<BITS>, grid, block, 0, s, st, (const uint32_t *)srcs[0],   \
                       (const char *)srcs[1], (const char *)srcs[2], (const uint32_t *)srcs[3],       \
                       (const char *)srcs[4], (const char *)srcs[5], nrows)
    switch (st.bits) {
        case 4: IMP(4); break;
        case 8: IMP(8); break;
        case 3: IMP(3); break;
        case 5: IMP(5); break;
        case 6: IMP(6); break;
        default: IMP(2); break;
    }
#undef IMP
    return hipGetLastError();
}

hipError_t launch_affine_quantize(const void *src, int64_t rows, int D, int gs, int bits, int dtype,
                                  uint32_t *wq, void *scales, void *biases, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    dim3 grid((unsigned)((rows + 3) / 4)), block(256);
    const int es = dtype == 2 ? 4 : 2;
#define CALL(DT, BITS)                                                                               \
    hipLaunchKernelGGL((affine_quantize_kernel<DT, BITS>), grid, block, 0, s, (const char *)src, rows, D, gs, \
                       wq, (char *)scales, (char *)biases, es)
    KV_DISPATCH_DT_BITS(dtype, bits, CALL);
#undef CALL
    return hipGetLastError();
}

hipError_t launch_affine_dequantize(const uint32_t *wq, const void *scales, const void *biases,
                                    int64_t rows, int D, int gs, int bits, int dtype, void *dst,
                                    hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    dim3 grid((unsigned)rows), block(128);
#define CALL(DT, BITS)                                                                               \
    hipLaunchKernelGGL((affine_dequantize_kernel<DT, BITS>), grid, block, 0, s, wq, (const char *)scales, \
                       (const char *)biases, rows, D, gs, (char *)dst)
    KV_DISPATCH_DT_BITS(dtype, bits, CALL);
#undef CALL
    return hipGetLastError();
}

// Plain fills and copies of plane memory run as kernels: they see virtual addresses only, so a
// range may span any number of separately mapped physical chunks, and no memset node ends up in
// a stream capture.  16-byte aligned pointers and sizes.
__global__ void __launch_bounds__(256) copy_bytes_kernel(u4v *dst, const u4v *src, size_t n16) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

// New pages: the memory behind them cleared and their entries put into the table, a thread to an entry, in one launch (a
// launch of its own for the entries held the next kernel up by 3 us).  `dst` may be null: entries only.
__global__ void __launch_bounds__(256) set_pages_kernel(u4v *dst, size_t n16, PageEntry *pt, int first, int count, PageEntry base, size_t sk, size_t sv,
                                                        size_t sksb, size_t svsb) {
    const size_t stride = (size_t)gridDim.x * 256, tid = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (size_t i = tid; i < (size_t)count; i += stride) {
        PageEntry e;
        e.k = base.k + i * sk;
        e.v = base.v + i * sv;
        e.ksb = base.ksb ? base.ksb + i * sksb : nullptr;
        e.vsb = base.vsb ? base.vsb + i * svsb : nullptr;
        pt[first + i] = e;
    }
    for (size_t i = tid; i < n16; i += stride) dst[i] = u4v{0u, 0u, 0u, 0u};
}

// grid (pages, 4 planes): the [BH] cells of one plane of one page, 16 bytes per thread and step
__global__ void __launch_bounds__(256) copy_pages_kernel(Store src, Store dst) {
    const PageEntry a = src.pt[blockIdx.x], b = dst.pt[blockIdx.x];
    const int plane = blockIdx.y;
    const char *from = plane == 0 ? a.k : plane == 1 ? a.v : plane == 2 ? a.ksb : a.vsb;
    char *to = plane == 0 ? b.k : plane == 1 ? b.v : plane == 2 ? b.ksb : b.vsb;
    const size_t cell = plane == 0 ? src.k_cell : plane == 1 ? src.v_cell : plane == 2 ? src.ksb_cell : src.vsb_cell;
    const size_t n16 = (size_t)src.BH * cell / 16;
    for (size_t i = threadIdx.x; i < n16; i += 256) reinterpret_cast<u4v *>(to)[i] = reinterpret_cast<const u4v *>(from)[i];
}

hipError_t launch_set_pages(void *clear, size_t bytes, PageEntry *pt, int first, int count, PageEntry base, const size_t stride[4], hipStream_t s) {
    if (count <= 0) return hipSuccess;
    if (((uintptr_t)clear | bytes) & 15) return hipErrorInvalidValue;
    const size_t n16 = clear ? bytes / 16 : 0;
    const unsigned grid = (unsigned)std::min<size_t>((std::max(n16, (size_t)count) + 255) / 256, 256 * 16);
    hipLaunchKernelGGL(set_pages_kernel, dim3(grid), dim3(256), 0, s, static_cast<u4v *>(clear), n16, pt, first, count, base, stride[0], stride[1],
                       stride[2], stride[3]);
    return hipGetLastError();
}

hipError_t launch_copy_pages(const Store &src, const Store &dst, int pages, hipStream_t s) {
    if (pages <= 0) return hipSuccess;
    hipLaunchKernelGGL(copy_pages_kernel, dim3(pages, src.bits ? 4 : 2), dim3(256), 0, s, src, dst);
    return hipGetLastError();
}

hipError_t launch_copy_bytes(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    if (((uintptr_t)dst | (uintptr_t)src | bytes) & 15) return hipErrorInvalidValue;
    const size_t n16 = bytes / 16;
    const unsigned grid = (unsigned)std::min<size_t>((n16 + 255) / 256, 256 * 16);
    hipLaunchKernelGGL(copy_bytes_kernel, dim3(grid), dim3(256), 0, s, static_cast<u4v *>(dst), static_cast<const u4v *>(src), n16);
    return hipGetLastError();
}

// Dense rows of one pitch into dense rows of another: the common prefix of every row is copied, what is left of a
// wider destination row is zero-filled.  (How arrays of a head size the tuned kernels are not built for are widened
// to the size the cache stores, and narrowed again on the way out.)
template <typename U>
__global__ void __launch_bounds__(256) repitch_rows_kernel(U *dst, uint32_t dst_units, const U *src, uint32_t src_units, size_t rows) {
    const size_t total = rows * dst_units;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const size_t row = i / dst_units;
        const uint32_t u = (uint32_t)(i - row * dst_units);
        dst[i] = u < src_units ? src[row * src_units + u] : (U)0;
    }
}

hipError_t launch_repitch_rows(void *dst, size_t dst_pitch, const void *src, size_t src_pitch, size_t rows, hipStream_t s) {
    if (rows == 0 || dst_pitch == 0) return hipSuccess;
    if ((dst_pitch | src_pitch) & 1) return hipErrorInvalidValue;
    const bool words = ((dst_pitch | src_pitch) & 3) == 0;
    const size_t units = rows * (dst_pitch / (words ? 4 : 2));
    const unsigned blocks = (unsigned)std::min<size_t>((units + 255) / 256, 4096);
    if (words)
        hipLaunchKernelGGL(repitch_rows_kernel<uint32_t>, dim3(blocks), dim3(256), 0, s, (uint32_t *)dst, (uint32_t)(dst_pitch / 4),
                           (const uint32_t *)src, (uint32_t)(src_pitch / 4), rows);
    else
        hipLaunchKernelGGL(repitch_rows_kernel<uint16_t>, dim3(blocks), dim3(256), 0, s, (uint16_t *)dst, (uint32_t)(dst_pitch / 2),
                           (const uint16_t *)src, (uint32_t)(src_pitch / 2), rows);
    return hipGetLastError();
}

hipError_t launch_mask_materialize(const kvhip_mask_plan_t &plan, uint8_t *dst, hipStream_t s) {
    if (plan.cols <= 0) return hipSuccess;
    dim3 grid((plan.cols + 255) / 256, plan.rolled ? 1 : (plan.rows < 1024 ? plan.rows : 1024)), block(256);
    hipLaunchKernelGGL(mask_materialize_kernel, grid, block, 0, s, plan, dst);
    return hipGetLastError();
}

}  // namespace kvhip
