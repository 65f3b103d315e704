// Quantize-on-append of many rows by 64-token tiles, whole ones and the partial ones at either end (from 3 to 14 rows up:
// `quant_tile_rows`): the element functions, the tile body and its two kernels, and the launchers of one code width
// (instantiated per width in kvhip_io.hip and kvhip_quant_tile_other.hip).
#pragma once
#include "kvhip_rope.hpp"

namespace kvhip {

namespace {

// ---- 64-token tiles (prompt-sized appends) -----------------------------------------------
// The per-row kernels above fetch one element per lane and wait for every row in turn; for
// many rows that is bound by load latency.  Here a workgroup takes one tile of one
// (batch, kv-head): every thread first requests all of its 16-byte chunks of the 64 new K and
// V rows, then quantizes / copies eight elements at a time.  Values, rounding and the
// rotation are those of the per-row kernels (the same element functions).
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// Eight elements of a row from the 16-byte chunk `raw` at d0, rotated when the chunk lies inside the rotary range.
template <int DT>
__device__ __forceinline__ void unpack8(const u4v &raw, const char *row, int d0, const RopeDev &rope, const float *inv_s, int pos,
                                        float (&w)[8]) {
    if (rope.dims > 0 && d0 < rope.dims) {
        if (rope.vec) {
            rope_chunk<DT>(rope, inv_s, row, d0, pos, raw, w);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = rope_elem<DT, true>(rope, row, d0 + j, pos);
        }
        return;
    }
    chunk_unpack<DT>(raw, w);
}

// Codes of the eight elements a thread holds, as integer-valued floats in [0, 2^BITS - 1], from
// the parameters of their group; `inv` is the hardware reciprocal of `scale`.
// code = rint((w - bias) / scale), clamped.  The quotient is first formed with the reciprocal
// (one ulp): product and reciprocal together put it within 2^-22 relative, so within 2^-14
// absolute (|quotient| <= 2^8), of the correctly rounded quotient, which can only change the
// rounded integer when the quotient sits that close to a half-integer.  Those elements (about
// one in 10^4) are redone with the exact division, so the codes are the reference's bit for bit.
// INVARIANT for anyone who edits this: the guard band (0.5 - 0.4999 = 1e-4) must stay above the
// largest error the fast quotient can have, which grows with the quotient: at |quotient| = 255 the
// reciprocal's one ulp plus the product's rounding come to about 4.6e-5.  Widening the code range
// (more than 8 bits) or replacing v_rcp_f32 by something less accurate needs a wider band; the
// known answers at 254.5 (tests/quantizer_kats.py, scale 3/256) and the tie stress in
// tests/test_gpu_cache.py fail if the band is too narrow.
template <int BITS>
__device__ __forceinline__ void codes8(const float (&w)[8], float scale, float bias, float inv, float (&q)[8]) {
    const float nb = (float)((1 << BITS) - 1);
    float dev = 0.0f;  // largest distance of a quotient from its rounded integer
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float r = __fmul_rn(__fsub_rn(w[j], bias), inv);
        const float c = rintf(r);
        dev = fmaxf(dev, fabsf(r - c));
        q[j] = fminf(fmaxf(c, 0.0f), nb);
    }
    if (dev > 0.4999f) {
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = (float)affine_code(w[j], scale, bias, nb);
    }
}

// `v` of the lane whose number is byte_addr / 4
__device__ __forceinline__ float lane_value(int byte_addr, float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(byte_addr, __builtin_bit_cast(int, v)));
}

// Four integer-valued floats in [0, 255] as the bytes of one word, first value lowest.
__device__ __forceinline__ uint32_t pack_bytes(float a, float b, float c, float d) {
    uint32_t w = __builtin_amdgcn_cvt_pk_u8_f32(a, 0, 0);
    w = __builtin_amdgcn_cvt_pk_u8_f32(b, 1, w);
    w = __builtin_amdgcn_cvt_pk_u8_f32(c, 2, w);
    return __builtin_amdgcn_cvt_pk_u8_f32(d, 3, w);
}
// Four integer-valued floats in [0, 15] as the nibbles of a 16-bit value, first value lowest
// (the sums stay below 2^16, so float32 arithmetic is exact).
__device__ __forceinline__ uint32_t pack_nibbles(float a, float b, float c, float d) {
    return (uint32_t)__builtin_fmaf(d, 4096.0f, __builtin_fmaf(c, 256.0f, __builtin_fmaf(b, 16.0f, a)));
}
// (scale, bias) of one group as the pair of 16-bit values the cache holds
template <int DT> __device__ __forceinline__ uint32_t pack_scale_bias(float scale, float bias) {
    if (DT == 0)
        return (uint32_t)__half_as_ushort(__float2half_rn(scale)) | ((uint32_t)__half_as_ushort(__float2half_rn(bias)) << 16);
    return (uint32_t)Elem<1>::bits(scale) | ((uint32_t)Elem<1>::bits(bias) << 16);
}

// One workgroup of NT threads: rows src0 .. src0 + n - 1 go to slots slot0 .. slot0 + n - 1, which may start
// and end inside a tile; 16-bit dtypes.
// GL = group size / 8 lanes share a quantization group; ROPE = false carries no rotation code.
// A thread holds 16-byte chunks of rows (a "chunk-instance" each), up to four at a
// time.  The extrema of every chunk-instance are reduced over the lanes of its group; then the
// affine parameters -- four exact divisions, the costly part -- are worked out once per group
// instead of once per lane: lane j of a group takes chunk-instance j (and j + GL, ...), writes
// that group's (scale, bias) pair, and the other lanes fetch bias and reciprocal from it.
// (Keys and values of a whole tile in one workgroup: 512 rows of
// 8 heads x 128 with the queries of 32, 13.3 us; the conversion of 5000 rows of 16 (batch, head) pairs 23.9 us.)
// PAGED: the 64 rows are tile `l_t / 64` of the full-precision page store `src` (a cache being
// converted) instead of rows of dense arrays: K chunks are read from the interleaved tile where
// they lie, the V tile (stored by column) is turned back into rows through LDS.
// SIDE: 1 the keys, 2 the values (NC being that side's head size by 32).  A workgroup takes TOK tokens of a tile, from
// token tok0 on, and COLS columns from col0 on: keys, which no column order asks for whole tiles of, go in pieces of few
// tokens, values in whole tiles of up to 128 columns.
template <int DT, int BITS, int NC, int GL, bool ROPE, bool PAGED, int SIDE, int NT, int TOK, int COLS>
__device__ __forceinline__ void append_quant_tile_body(const Store &st, const Store &src, const char *keys, const char *values,
                                                       int L, int src0, int slot0, int n, const RopeDev &rope, int tile, int tok0, int col0) {
    constexpr int D = 32 * NC;
    constexpr int GS = 8 * GL;
    constexpr int TPR = COLS / 8;   // threads per row
    constexpr int VP = COLS + 8;    // byte pitch of a token's V codes in LDS
    constexpr bool DO_K = SIDE == 1, DO_V = SIDE == 2;
    static_assert(COLS % GS == 0 && (DO_K ? COLS == D : TOK == TILE), "whole groups; whole rows of keys, whole tiles of values");
    constexpr int NCH = TOK * TPR / NT;  // chunks of a thread
    static_assert(NCH * NT == TOK * TPR, "every thread holds as many");
    constexpr int EB = NCH % 4 == 0 ? 4 : NCH % 3 == 0 ? 3 : NCH % 2 == 0 ? 2 : 1;  // chunks per batch
    constexpr int SH = EB == 3 ? 4 : EB;  // lanes of a group that work out parameters, one chunk-instance each
    // a row's TPR threads: where NT is a multiple of TPR the rows of a thread's chunks are NT / TPR apart and
    // its columns the same; at D = 96 (12 threads per row) row and column are worked out per chunk
    constexpr bool EVEN = NT % TPR == 0;
    constexpr bool GEN = BITS != 4 && BITS != 8;  // 2, 3, 5, 6 bits: codes as a plain bit stream, K rows and V tile rows alike
    // the source V tile as stored and, once every thread has its chunks of it, the codes
    __shared__ __attribute__((aligned(16))) uint8_t vcodes[!DO_V ? 16 : PAGED ? TILE * COLS * 2 : TILE * VP];
    __shared__ __attribute__((aligned(16))) uint8_t kcodes[GEN && DO_K ? TOK * D * BITS / 8 : 16];  // the K rows as stored
    __shared__ float inv_s[ROPE ? D / 2 : 1];
    const int bh = blockIdx.y;
    const int slot_t = (slot0 & ~(TILE - 1)) + tile * TILE;
    const int l_t = src0 + slot_t - slot0;  // the row in the tile's first slot (before the first new row: t_lo > 0)
    // tokens [t_lo, t_hi) of the tile are new.  The threads of the others repeat the nearest new row, which keeps their
    // loads inside the arrays, and write nothing.
    const int t_lo = PAGED ? 0 : max(slot0 - slot_t, 0), t_hi = min(PAGED ? TILE : slot0 + n - slot_t, tok0 + TOK);
    if (DO_K && (tok0 >= t_hi || tok0 + TOK <= t_lo)) return;  // (workgroup-uniform)
    const bool whole = t_lo <= tok0 && t_hi == tok0 + TOK;
    const char *base = PAGED ? nullptr : (DO_K ? keys : values) + (((ptrdiff_t)bh * L + l_t) * D + col0) * 2;
    u4v raw[NCH];
    if constexpr (PAGED) {
        const char *kt = k_cell_ptr(src, bh, l_t) + kfp_off(src, l_t, 0);   // tile start: [chunk][token][16 B]
        const char *vt = v_cell_ptr(src, bh, l_t) + vfp_off(src, l_t, 0);   // tile start: [8-token chunk][column][16 B]
#pragma unroll
        for (int e = 0; e < NCH; ++e) {
            const int c = e * NT + threadIdx.x;
            if constexpr (DO_K) raw[e] = *reinterpret_cast<const u4v *>(kt + ((size_t)(c % TPR) * TILE + tok0 + c / TPR) * 16);
            if constexpr (DO_V) *reinterpret_cast<u4v *>(vcodes + (size_t)c * 16) = *reinterpret_cast<const u4v *>(vt + ((size_t)(c / COLS) * D + col0 + c % COLS) * 16);
        }
        if constexpr (DO_V) __syncthreads();
#pragma unroll
        for (int e = 0; e < (DO_V ? NCH : 0); ++e) {
            const int c = e * NT + threadIdx.x;
            const int r = c / TPR, dd = (c - r * TPR) * 8;
            const uint16_t *col = reinterpret_cast<const uint16_t *>(vcodes) + ((size_t)(r >> 3) * COLS + dd) * 8 + (r & 7);
            uint32_t u[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = (uint32_t)col[(2 * j) * 8] | ((uint32_t)col[(2 * j + 1) * 8] << 16);
            raw[e] = u4v{u[0], u[1], u[2], u[3]};
        }
        if constexpr (DO_V) __syncthreads();
    } else {
#pragma unroll
        for (int e = 0; e < NCH; ++e) {
            const int c = e * NT + threadIdx.x, r = tok0 + c / TPR;
            raw[e] = *reinterpret_cast<const u4v *>(base + ((ptrdiff_t)min(max(r, t_lo), t_hi - 1) * D + (c % TPR) * 8) * 2);
        }
    }
    if constexpr (ROPE) {
        rope_inv_table(rope, inv_s);
        __syncthreads();
    }
    const float nb = (float)((1 << BITS) - 1);
    const int lane = threadIdx.x & 63;
    const int pos = lane & (GL - 1);            // place in the group
    const int psel = pos & (SH - 1);
    const int gbase4 = (lane & ~(GL - 1)) * 4;  // byte address (lane number x 4) of the group's first lane
    const int r_t = tok0 + threadIdx.x / TPR;   // row of this thread's chunk 0; chunk e lies NT / TPR rows further
    const int d0_t = (threadIdx.x % TPR) * 8;   // (columns count from col0)
    auto row_of = [&](int e) { return EVEN ? r_t + e * (NT / TPR) : tok0 + (e * NT + (int)threadIdx.x) / TPR; };
    auto col_of = [&](int e) { return EVEN ? d0_t : ((e * NT + (int)threadIdx.x) % TPR) * 8; };
    const int page_off = (slot_t & (PAGE - 1));
    const ptab entry = page_table(st) + (slot_t >> PAGE_SHIFT);  // a tile lies inside one page
    const PageEntry page{entry->k, entry->ksb, entry->v, entry->vsb};
#pragma unroll
    for (int e0 = 0; e0 < NCH; e0 += EB) {
        float w[EB][8], mn[EB], mx[EB];
#pragma unroll
        for (int i = 0; i < EB; ++i) {
            const int e = e0 + i;
            const int d0 = col_of(e);
            if constexpr (ROPE && DO_K) {
                const int r = min(max(row_of(e), t_lo), t_hi - 1);
                unpack8<DT>(raw[e], base + (size_t)r * D * 2, d0, rope, inv_s, rope_pos(rope, bh, l_t + r), w[i]);
            } else {
                chunk_unpack<DT>(raw[e], w[i]);
            }
            float a = w[i][0], b = w[i][0];
#pragma unroll
            for (int j = 1; j < 8; ++j) {
                a = fminf(a, w[i][j]);
                b = fmaxf(b, w[i][j]);
            }
            group_minmax_dpp<GL>(a, b);
            mn[i] = a;
            mx[i] = b;
        }
        float sc, bi, iv;  // of chunk-instance psel (the fourth of three: the first again, which nobody asks for)
        {
            float a = mn[0], b = mx[0];
#pragma unroll
            for (int j = 1; j < EB; ++j) {
                a = psel == j ? mn[j] : a;
                b = psel == j ? mx[j] : b;
            }
            affine_params(a, b, nb, sc, bi);
            iv = __builtin_amdgcn_rcpf(sc);
            const int e = e0 + psel, t_sb = row_of(e);
            if (pos < SH && psel < EB && t_sb >= t_lo && t_sb < t_hi) {
                const int row = page_off + t_sb;
                char *sb = DO_V ? page.vsb + (size_t)bh * st.vsb_cell + (size_t)row * st.vsb_row
                                : page.ksb + (size_t)bh * st.ksb_cell + (size_t)row * st.ksb_row;
                reinterpret_cast<uint32_t *>(sb)[(col0 + col_of(e)) / GS] = pack_scale_bias<DT>(sc, bi);
            }
        }
#pragma unroll
        for (int i = 0; i < EB; ++i) {
            const int e = e0 + i;
            const int r = row_of(e), d0 = col_of(e);
            const int src = gbase4 + i * 4;
            const float scale = lane_value(src, sc);
            const float bias = lane_value(src, bi);
            const float inv = lane_value(src, iv);
            float q[8];
            codes8<BITS>(w[i], scale, bias, inv, q);
            if constexpr (DO_K) {
                // ---- K: packed words in natural order --------------------------------------------
                uint32_t *kw = reinterpret_cast<uint32_t *>(page.k + (size_t)bh * st.k_cell + (size_t)(page_off + r) * st.k_row);
                if (!GEN && (r < t_lo || r >= t_hi)) continue;
                if constexpr (BITS == 4) {
                    kw[d0 / 8] = pack_nibbles(q[0], q[1], q[2], q[3]) | (pack_nibbles(q[4], q[5], q[6], q[7]) << 16);
                } else if constexpr (BITS == 8) {
                    *reinterpret_cast<uint2 *>(kw + d0 / 4) =
                        make_uint2(pack_bytes(q[0], q[1], q[2], q[3]), pack_bytes(q[4], q[5], q[6], q[7]));
                } else {
                    // eight codes are BITS whole bytes of the row's bit stream; the tile's K rows follow each other
                    // in the page, so they are collected in LDS and leave as 16-byte chunks below
                    uint64_t bits8 = 0;
#pragma unroll
                    for (int j = 0; j < 8; ++j) bits8 |= (uint64_t)(uint32_t)q[j] << (j * BITS);
                    uint8_t *kb = &kcodes[(r - tok0) * (D * BITS / 8) + (d0 / 8) * BITS];
#pragma unroll
                    for (int j = 0; j < BITS; ++j) kb[j] = (uint8_t)(bits8 >> (8 * j));
                }
            } else {
                // ---- V: codes as bytes, transposed below -----------------------------------------
                *reinterpret_cast<uint2 *>(&vcodes[r * VP + d0]) =
                    make_uint2(pack_bytes(q[0], q[1], q[2], q[3]), pack_bytes(q[4], q[5], q[6], q[7]));
            }
        }
    }
    if constexpr (GEN && DO_K) {
        __syncthreads();
        char *kt = page.k + (size_t)bh * st.k_cell + (size_t)(page_off + tok0) * st.k_row;  // TOK rows of D BITS / 8 bytes, contiguous
        if (whole) {
            for (int c = threadIdx.x; c < TOK * D * BITS / 8 / 16; c += NT)
                *reinterpret_cast<u4v *>(kt + (size_t)c * 16) = *reinterpret_cast<const u4v *>(&kcodes[c * 16]);
        } else {  // (rows are whole words: D is a multiple of 32)
            constexpr int RW = D * BITS / 32;
            for (int c = max(t_lo - tok0, 0) * RW + threadIdx.x; c < min(t_hi - tok0, TOK) * RW; c += NT)
                reinterpret_cast<uint32_t *>(kt)[c] = reinterpret_cast<const uint32_t *>(kcodes)[c];
        }
    }
    if constexpr (!DO_V) return;
    __syncthreads();
    char *cell = page.v + (size_t)bh * st.v_cell + v_row_off(st, slot_t, col0);
    if constexpr (GEN) {
        // a transposed row is the bit stream of its 64 tokens' codes: 32 tokens fill BITS words, which a thread
        // assembles with every shift a constant; consecutive threads write consecutive words.  (A word to a thread, whose
        // first token depends on the word: 3 bits, 2048 rows of 64 pairs x 128: 33.9 us for 24.0.)
        for (int c = threadIdx.x; c < COLS * 2; c += NT) {
            const int d = c >> 1, t0 = (c & 1) * 32;
            uint32_t word[BITS] = {}, mine[BITS] = {};  // (mine: the bits of new tokens)
#pragma unroll
            for (int t = 0; t < 32; ++t) {
                const uint32_t code = vcodes[(t0 + t) * VP + d];
                const uint32_t ones = t0 + t >= t_lo && t0 + t < t_hi ? (1u << BITS) - 1u : 0u;
                const int w = t * BITS / 32, sh = t * BITS % 32;
                word[w] |= code << sh;
                mine[w] |= ones << sh;
                if (sh + BITS > 32) {
                    word[w + 1] |= code >> (32 - sh);
                    mine[w + 1] |= ones >> (32 - sh);
                }
            }
            uint32_t *p = reinterpret_cast<uint32_t *>(cell + (size_t)d * (TILE * BITS / 8)) + (c & 1) * BITS;
#pragma unroll
            for (int w = 0; w < BITS; ++w) {
                if (mine[w] == 0xffffffffu) p[w] = word[w];
                else if (mine[w] != 0) p[w] = (p[w] & ~mine[w]) | (word[w] & mine[w]);
            }
        }
        return;
    }
    // Two words of the transposed rows of four columns to a thread: tokens are read four codes at a time, nibbles paired
    // with the bytes still side by side and the bytes turned by permutes, in the order v_bitpos gives.  Consecutive threads
    // continue the rows.  (A row's 16 bytes to a thread, code by code: 4 bits, 2048 rows of 64 pairs x 128, 19.5 us for
    // 19.2; 8 bits 23.8 for 21.5.)
    constexpr int TPW = 32 / BITS;        // tokens per word
    constexpr int CPR = TILE / TPW / 2;   // 8-byte chunks per row
    for (int c = threadIdx.x; c < COLS / 4 * CPR; c += NT) {
        const int d = c / CPR * 4, q = c % CPR;
        uint32_t out[4][2];
#pragma unroll
        for (int wi = 0; wi < 2; ++wi) {
            uint32_t in[TPW];  // one token's codes of the four columns
#pragma unroll
            for (int t = 0; t < TPW; ++t) in[t] = *reinterpret_cast<const uint32_t *>(&vcodes[((2 * q + wi) * TPW + t) * VP + d]);
            uint32_t byte[4];  // byte j of the four columns' words
            if constexpr (BITS == 4) {
                byte[0] = in[0] | (in[2] << 4), byte[1] = in[4] | (in[6] << 4);
                byte[2] = in[1] | (in[3] << 4), byte[3] = in[5] | (in[7] << 4);
            } else {
                byte[0] = in[0], byte[1] = in[2], byte[2] = in[1], byte[3] = in[3];
            }
            const uint32_t a01 = __builtin_amdgcn_perm(byte[1], byte[0], 0x05010400), a23 = __builtin_amdgcn_perm(byte[1], byte[0], 0x07030602);
            const uint32_t b01 = __builtin_amdgcn_perm(byte[3], byte[2], 0x05010400), b23 = __builtin_amdgcn_perm(byte[3], byte[2], 0x07030602);
            out[0][wi] = __builtin_amdgcn_perm(b01, a01, 0x05040100);
            out[1][wi] = __builtin_amdgcn_perm(b01, a01, 0x07060302);
            out[2][wi] = __builtin_amdgcn_perm(b23, a23, 0x05040100);
            out[3][wi] = __builtin_amdgcn_perm(b23, a23, 0x07060302);
        }
        uint32_t *dst = reinterpret_cast<uint32_t *>(cell + (size_t)d * (TILE * BITS / 8) + 8 * q);
        constexpr int RW = TILE * BITS / 32;  // words from row to row
        if (whole) {
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<uint2 *>(dst + j * RW) = make_uint2(out[j][0], out[j][1]);
        } else {
#pragma unroll
            for (int wi = 0; wi < 2; ++wi) {
                uint32_t mine = 0;  // the bits of new tokens in this word
#pragma unroll
                for (int tt = 0; tt < TPW; ++tt) {
                    const int t = (2 * q + wi) * TPW + tt;
                    if (t >= t_lo && t < t_hi) mine |= ((1u << BITS) - 1u) << (v_bitpos<BITS>(t) & 31);
                }
                if (mine == 0) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t *p = dst + j * RW + wi;
                    *p = mine == 0xffffffffu ? out[j][wi] : (*p & ~mine) | (out[j][wi] & mine);
                }
            }
        }
    }
}

// How a tile's work is cut: workgroups of NT threads, K in pieces of TOK tokens, V in blocks of COLS columns.  Rows that
// turn: few chunks to a thread, each of eight angles (2048 rows of 64 (batch, head) pairs, 4 bits: x 128 38.7 us with keys
// and values of a tile in one workgroup, 33.2 so; 32 pairs x 256 26.2 and 19.1).  Others: the chunks of a group share the
// lanes that work out parameters, so up to four to a thread (x 128 20.5 and 19.2 us; 8 bits 23.1 and 21.5; 3 bits 30.3 and
// 24.0).  With 128 threads and eight chunks it was 22.6.  PAGED in blocks of 64 columns, whose LDS -- the workgroups of K
// are charged it too -- decides how many fit a CU (the conversion above: 15.5 us, 25.2 with blocks of 128 columns).
// (NC = 3, 6: 192 threads, of which every row takes twelve or twenty-four.)
template <int NC, int GL, int SIDE, bool ROPE, bool PAGED> struct QuantTile {
    static constexpr int NT = NC % 3 == 0 ? 192 : 256;
    static constexpr int TOK = ROPE ? (NC == 2 ? 32 : NC <= 6 ? 16 : 8) : NC >= 6 ? 32 : TILE;
    static constexpr int COLS = NC == 3 ? 96 : PAGED ? (GL > 8 ? 128 : 64) : NC > 4 ? 128 : 32 * NC;
    static constexpr int KP = SIDE == 2 ? 0 : TILE / TOK, VP = SIDE == 1 ? 0 : 32 * NC / COLS;
    static constexpr int PIECES = KP + VP;
};
// piece `piece` of tile `tile`: the values first, whose workgroups take the longer
template <int DT, int BITS, int NC, int GL, bool ROPE, bool PAGED, int SIDE>
__device__ __forceinline__ void quant_tile_piece(const Store &st, const Store &src, const char *keys, const char *values, int L, int src0, int slot0,
                                                 int n, const RopeDev &rope) {
    using Q = QuantTile<NC, GL, SIDE, ROPE, PAGED>;
    const int tile = blockIdx.x / Q::PIECES, piece = blockIdx.x - tile * Q::PIECES;
    if constexpr (SIDE != 1) {
        if (SIDE == 2 || piece < Q::VP) {
            append_quant_tile_body<DT, BITS, NC, GL, false, PAGED, 2, Q::NT, TILE, Q::COLS>(st, src, keys, values, L, src0, slot0, n, rope, tile, 0,
                                                                                            piece * Q::COLS);
            return;
        }
    }
    if constexpr (SIDE != 2)
        append_quant_tile_body<DT, BITS, NC, GL, ROPE, PAGED, 1, Q::NT, Q::TOK, 32 * NC>(st, src, keys, values, L, src0, slot0, n, rope, tile,
                                                                                         (piece - Q::VP) * Q::TOK, 0);
}

// SIDE: 0 keys and values of one head size 32 NC; 1 the keys alone, 2 the values alone (caches whose keys and
// values differ in head size take one launch for each, NC being that side's).
template <int DT, int BITS, int NC, int GL, bool ROPE, int SIDE = 0>
__global__ void __launch_bounds__((QuantTile<NC, GL, SIDE, ROPE, false>::NT))
append_quant_tile_kernel(Store st, const char *keys, const char *values, int L, int src0, int slot0, int n, RopeDev rope) {
    if constexpr (ROPE) {
        if ((int)blockIdx.y >= st.BH) {  // queries of the same forward
            __shared__ float q_inv_s[NC * 16];
            rope_queries_ride<DT>(rope, st.BH, q_inv_s);
            return;
        }
    }
    quant_tile_piece<DT, BITS, NC, GL, ROPE, false, SIDE>(st, st, keys, values, L, src0, slot0, n, rope);
}

// grid (pieces of tiles, BH): the tiles of the full-precision store `src` into the same slots of `st`
template <int DT, int BITS, int NC, int GL, int SIDE = 0>
__global__ void __launch_bounds__((QuantTile<NC, GL, SIDE, false, true>::NT)) requant_tile_kernel(Store st, Store src) {
    quant_tile_piece<DT, BITS, NC, GL, false, true, SIDE>(st, src, nullptr, nullptr, 0, 0, 0, 0, RopeDev());
}

// Which stores the tile kernels take: 16-bit dtypes, group size 32 / 64 / 128 dividing the head size; keys and
// values of one head size in 64 / 96 / 128 / 256 (one launch), or keys of 192 with values of 128 (a launch for
// each side; 4- and 8-bit codes, group size 32 or 64).
inline bool quant_tiles_one_launch(const Store &st) {
    return st.es == 2 && st.Dk == st.Dv && (st.Dk == 64 || st.Dk == 96 || st.Dk == 128 || st.Dk == 256) &&
           (st.gs == 32 || st.gs == 64 || st.gs == 128) && st.Dk % st.gs == 0;
}
inline bool quant_tiles_two_sided(const Store &st) {
    return st.es == 2 && st.Dk == 192 && st.Dv == 128 && (st.bits == 4 || st.bits == 8) && (st.gs == 32 || st.gs == 64);
}

// The launches of one code width.  PAGED = false: `n` dense rows from row a0 on into the slots from b0 on; PAGED = true:
// the tiles that hold rows [0, n) of the full-precision store `src` into the same slots.
// TWO_SIDED: also the instances for keys of 192 with values of 128.
template <int DT, int BITS, int NC, int GL, int SIDE, bool PAGED>
void launch_quant_tile_instance(const Store &st, const Store &src, const void *keys, const void *values, int L, int a0,
                                int b0, int n, hipStream_t s, const RopeDev &r) {
    const int tiles = (PAGED ? (n + TILE - 1) : ((b0 & (TILE - 1)) + n + TILE - 1)) / TILE;
    if constexpr (PAGED) {
        using Q = QuantTile<NC, GL, SIDE, false, true>;
        hipLaunchKernelGGL((requant_tile_kernel<DT, BITS, NC, GL, SIDE>), dim3(tiles * Q::PIECES, st.BH), dim3(Q::NT), 0, s, st, src);
    } else if (r.dims > 0 && SIDE != 2) {
        using Q = QuantTile<NC, GL, SIDE, true, false>;
        const int gx = tiles * Q::PIECES;
        hipLaunchKernelGGL((append_quant_tile_kernel<DT, BITS, NC, GL, true, SIDE>), dim3(gx, st.BH + rope_ride_rows(r, gx, st.es, Q::NT)), dim3(Q::NT), 0, s, st,
                           (const char *)keys, (const char *)values, L, a0, b0, n, r);
    } else {
        using Q = QuantTile<NC, GL, SIDE, false, false>;
        hipLaunchKernelGGL((append_quant_tile_kernel<DT, BITS, NC, GL, false, SIDE>), dim3(tiles * Q::PIECES, st.BH), dim3(Q::NT), 0, s, st,
                           (const char *)keys, (const char *)values, L, a0, b0, n, r);
    }
}

template <int DT, int BITS, bool TWO_SIDED, bool PAGED>
hipError_t launch_quant_tiles_dt(const Store &st, const Store &src, const void *keys, const void *values, int L, int a0,
                                 int b0, int n, hipStream_t s, const RopeDev &r) {
#define KV_TILE(NC, GL, SIDE) launch_quant_tile_instance<DT, BITS, NC, GL, SIDE, PAGED>(st, src, keys, values, L, a0, b0, n, s, r)
#define KV_TILE_GL(NC)                        \
    do {                                      \
        if (st.gs == 32) KV_TILE(NC, 4, 0);   \
        else if (st.gs == 64) KV_TILE(NC, 8, 0); \
        else KV_TILE(NC, 16, 0);              \
    } while (0)
    if (quant_tiles_one_launch(st)) {
        if (st.Dk == 64 && st.gs == 32) KV_TILE(2, 4, 0);
        else if (st.Dk == 64) KV_TILE(2, 8, 0);
        else if (st.Dk == 96) KV_TILE(3, 4, 0);
        else if (st.Dk == 128) KV_TILE_GL(4);
        else KV_TILE_GL(8);
        return hipGetLastError();
    }
    if constexpr (TWO_SIDED) {
        if (quant_tiles_two_sided(st)) {
            if (st.gs == 32) {
                KV_TILE(6, 4, 1);
                KV_TILE(4, 4, 2);
            } else {
                KV_TILE(6, 8, 1);
                KV_TILE(4, 8, 2);
            }
            return hipGetLastError();
        }
    }
#undef KV_TILE_GL
#undef KV_TILE
    return hipErrorInvalidValue;
}

template <int BITS, bool TWO_SIDED, bool PAGED>
hipError_t launch_quant_tiles_bits(const Store &st, const Store &src, const void *keys, const void *values, int L, int a0,
                                   int b0, int n, hipStream_t s, const RopeDev &r) {
    if (n <= 0) return hipSuccess;
    if (st.dtype == KVHIP_F16) return launch_quant_tiles_dt<0, BITS, TWO_SIDED, PAGED>(st, src, keys, values, L, a0, b0, n, s, r);
    if (st.dtype == KVHIP_BF16) return launch_quant_tiles_dt<1, BITS, TWO_SIDED, PAGED>(st, src, keys, values, L, a0, b0, n, s, r);
    return hipErrorInvalidValue;
}

}  // namespace

}  // namespace kvhip
