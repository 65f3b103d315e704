// Split-sequence decode attention on the matrix cores (gfx950).
//
// One workgroup (4 wavefronts) owns a contiguous span of physical slots of one
// (batch, kv-head) pair and leaves an unnormalised partial (max, sum, out[D]) per
// query row; a second small kernel merges the partials of all spans.  All query
// rows that share a kv head (r = Hq/Hkv heads times L new tokens, up to 16) are
// served from one pass over K and V, which are read from HBM exactly once.
//
// The contraction uses v_mfma_f32_4x4x4_16B_f16: sixteen independent 4x4x4 blocks
// per instruction.  With CBSZ=4 the A operand of ONE block (chosen by ABID) is
// broadcast to all sixteen, so the small operand (4 query rows / 4 probability
// rows) costs two registers while the large one (K, V) fills the B side:
//
//   QK^T  block b covers tokens 4b..4b+3: lane l supplies four head-dim elements
//         of token l's K row (B); the accumulator of lane l receives the scores of
//         token l for the 4 query rows.  The query operands of 16 successive steps
//         live in the 16 lane groups of one register pair; ABID picks the step.
//   PV    block b covers head-dim columns 4b..4b+3 (+64h): lane l supplies, for
//         column l, four consecutive tokens of the transposed V tile (B); the
//         probabilities of step s (tokens 4s..4s+3) sit in lane group s after a
//         4x4 transpose inside each quad of lanes and are broadcast with ABID = s.
//
// Packed codes become operands without a dequantize pass: a code masked in place
// is the fp16 subnormal code * 2^-24 (high nibbles: * 2^-20, compensated by
// operands pre-scaled by 1/16), which the matrix core multiplies exactly.  So
//   q . (scale*code + bias)            = scale * 2^24 * mfma(q, masked K words) + bias * sum(q)
//   sum_t p_t (scale_t*code_t + bias_t) = 2^24 * mfma(p*scale, masked V words) + sum_t p_t bias_t
#include <cstdlib>
#include <type_traits>
#include <utility>
#include <vector>

#include "kvhip_mask.hpp"
#include "kvhip_rope.hpp"
#include "kvhip_span_merge.hpp"
#include "kvhip_wave.hpp"

// piece buffers of the full-precision decode kernel (at most the D / 32 pieces of one tile)
#ifndef KVHIP_DECODE_FP_NBUF
#define KVHIP_DECODE_FP_NBUF(D, RG) 2
#endif

namespace kvhip {

namespace {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
union Op {  // one 4-element 16-bit operand
    h4 h;
    s4 s;
    uint32_t u[2];
};

constexpr int WAVES = 4;
constexpr float TWO24 = 16777216.0f;

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
// f(std::integral_constant<int, i>) for i = 0..N-1, fully unrolled with compile-time i
template <int N, class F> __device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int ABID> __device__ __forceinline__ f4 mfma444(const Op &a, const Op &b, f4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(a.h, b.h, c, 4, ABID, 0);
}
template <int ABID> __device__ __forceinline__ f4 mfma444_bf(const Op &a, const Op &b, f4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a.s, b.s, c, 4, ABID, 0);
}

__device__ __forceinline__ float uniform(float v) {  // v is the same in every lane
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ uint16_t f2h_bits(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
__device__ __forceinline__ uint32_t pack_h2(float lo, float hi) { return pk_h2(lo, hi); }

// value held by lane (l ^ 1) / (l ^ 2) of the same quad
__device__ __forceinline__ uint32_t quad_xor1(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ uint32_t quad_xor2(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);  // quad_perm [2,3,0,1]
}
// 4x4 transpose inside each quad: before, lane c holds x[i]; after, lane i holds in
// x[k] what lane k held in x[i].
__device__ __forceinline__ void quad_transpose(uint32_t x[4], int lane) {
    const bool b0 = lane & 1, b1 = lane & 2;
    {
        const uint32_t s01 = b0 ? x[0] : x[1], s23 = b0 ? x[2] : x[3];
        const uint32_t r01 = quad_xor1(s01), r23 = quad_xor1(s23);
        x[0] = b0 ? r01 : x[0];
        x[1] = b0 ? x[1] : r01;
        x[2] = b0 ? r23 : x[2];
        x[3] = b0 ? x[3] : r23;
    }
    {
        const uint32_t s02 = b1 ? x[0] : x[2], s13 = b1 ? x[1] : x[3];
        const uint32_t r02 = quad_xor2(s02), r13 = quad_xor2(s13);
        x[0] = b1 ? r02 : x[0];
        x[2] = b1 ? x[2] : r02;
        x[1] = b1 ? r13 : x[1];
        x[3] = b1 ? x[3] : r13;
    }
}

// load N consecutive dwords with the widest vector accesses
// (from device memory: a `gptr`, so that the loads are GLOBAL rather than FLAT ones)
template <int N> __device__ __forceinline__ void load_words(uint32_t *dst, gptr p) {
    if constexpr (N % 4 == 0) {
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            const kv_u4 v = ld_global<kv_u4>(p, i);
            dst[4 * i] = v.x; dst[4 * i + 1] = v.y; dst[4 * i + 2] = v.z; dst[4 * i + 3] = v.w;
        }
    } else if constexpr (N % 2 == 0) {
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const kv_u2 v = ld_global<kv_u2>(p, i);
            dst[2 * i] = v.x; dst[2 * i + 1] = v.y;
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) dst[i] = ld_global<uint32_t>(p, i);
    }
}

// ---- operand geometry --------------------------------------------------------------
// A "step" contracts 4 elements; one packed 32-bit word yields WSTEPS steps.
//   4 bit: 8 codes -> 2 steps taking nibbles (0,4,1,5) and (2,6,3,7); the last two
//          of each are high nibbles (value x16)
//   8 bit: 4 codes -> 1 step taking bytes (0,2,1,3)
template <int BITS> struct Geo;
template <> struct Geo<4> {
    static constexpr int WSTEPS = 2, EPW = 8;
    static __device__ __forceinline__ constexpr int elem(int h, int k) { return 2 * h + (k >> 1) + 4 * (k & 1); }
    static __device__ __forceinline__ constexpr bool hi(int k) { return k >= 2; }
    static __device__ __forceinline__ void unpack(uint32_t w, Op *o) {
        const uint32_t w8 = w >> 8;
        o[0].u[0] = w & 0x000f000fu;
        o[0].u[1] = w & 0x00f000f0u;
        o[1].u[0] = w8 & 0x000f000fu;
        o[1].u[1] = w8 & 0x00f000f0u;
    }
};
template <> struct Geo<8> {
    static constexpr int WSTEPS = 1, EPW = 4;
    static __device__ __forceinline__ constexpr int elem(int, int k) { return (k >> 1) + 2 * (k & 1); }
    static __device__ __forceinline__ constexpr bool hi(int) { return false; }
    static __device__ __forceinline__ void unpack(uint32_t w, Op *o) {
        o[0].u[0] = w & 0x00ff00ffu;
        o[0].u[1] = (w >> 8) & 0x00ff00ffu;
    }
};

// scale / bias of a (scale, bias) pair of a 16-bit dtype; the first also: the one element in the low half
template <int DT> __device__ __forceinline__ float pair_scale(uint32_t raw) {
    return DT == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)raw) : __uint_as_float(raw << 16);
}
template <int DT> __device__ __forceinline__ float pair_bias(uint32_t raw) {
    return DT == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(raw >> 16)) : __uint_as_float(raw & 0xffff0000u);
}

// One tile (64 slots) of raw operand data in registers; lane l owns token l of the tile
// for K and head-dim column l (+64h) for V.
template <int BITS, int D, int G> struct TileRegs {
    static constexpr int KW = D * BITS / 32;   // dwords of one K row
    static constexpr int VW = 64 * BITS / 32;  // dwords of one V tile row
    uint32_t k[KW];
    uint32_t v[D / 64][VW];
    uint32_t ksb[G], vsb[G];  // (scale, bias) pairs as stored: turned into floats where they are used, so that nothing waits for them before
    int row;    // presented row of this lane's token, -1 if none
    bool edge;  // wave-uniform: some token of the tile is dead or masked for some query row
};

// Hq / Hkv for at most MAX query heads to a kv head: comparisons in place of a division, which a step's first request would
// wait for (with those of the batch row and of the query rows' heads: 0.2 us of a launch).
template <int MAX> __device__ __forceinline__ int heads_of_a_kv_head(int Hq, int Hkv) {
    int r = 1;
#pragma unroll
    for (int i = 2; i <= MAX; ++i) r += Hq >= i * Hkv ? 1 : 0;
    return r;
}

// RG = groups of 4 query rows handled per pass (R <= 4 RG).  MM selects the mask code:
// 0 none (the tile loop is branch free), 1 index-only masks (causal / window, per-batch
// bounds preloaded: no memory access in the loop), 2 array masks (loads in the loop, which
// force conservative waits on the prefetch).  Slots map to presented rows one to one: only
// RotatingKVCache remaps slots, and it is never quantized.
// NW = wavefronts per workgroup: 4 (two workgroups per CU), or 8 when that lets one
// workgroup take the whole sequence of its (batch, kv-head) pair -- then the output rows are
// normalised and written here and no partial goes through memory.
// MODE 3: MM 0, with the step's rows still to be rotated.
template <int BITS, int D, int GS, int DT, int RG, int MODE, int NW>
__global__ void __launch_bounds__(NW * 64, NW == 4 ? 2 : 1)
decode_kernel(int tiles_total, int tiles_per_wg, int nsplit, typename DecodeArgs<MODE>::type a) {
    fetch_arguments(a, tiles_total, tiles_per_wg, nsplit);
    constexpr int MM = MODE == 3 ? 0 : MODE;
    constexpr bool rot = MODE == 3;
    using GEO = Geo<BITS>;
    constexpr int G = D / GS;      // quantization groups per row (1, 2 or 4)
    constexpr int NH = D / 64;     // 64-column halves of the output
    constexpr int NQA = D / 64;    // query operand register pairs (16 steps of 4 elements each)
    constexpr int RR = 4 * RG;     // query rows carried
    // Group size 32: the 64 columns a PV instruction covers lie in two groups, and the probability
    // operand (which carries the V scale) is the same for every lane.  Each V step is therefore
    // issued twice, once with either group's operand, into two accumulators; lanes 0-31 keep the
    // first, lanes 32-63 the second.
    constexpr bool HALF = GS < 64;
    constexpr int NO2 = HALF ? D / 64 : 1;  // second accumulators (one dummy when unused)
    using T = TileRegs<BITS, D, G>;
    const Store &st = a.st;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    const int blk = lane >> 2, qi = lane & 3;  // lane group (MFMA block) and position in it
    int bh = blockIdx.y;
    const int split = blockIdx.x;
    int b = MM == 0 ? 0 : bh / a.Hkv;  // (without a mask nothing asks for it)
    [[maybe_unused]] const int hk = bh - b * a.Hkv;
    size_t part_slot = (size_t)bh * nsplit + split;  // where this workgroup's partial goes
    [[maybe_unused]] RaggedSpan span;
    [[maybe_unused]] int wid = 0;
    if constexpr (MM == 1) {
        if (__builtin_expect(tiles_per_wg < 0, 0)) {  // a ragged batch that shares its spans out (behind the rest of the kernel)
            wid = b * nsplit + split;
            span = ragged_span(a.mask, a.B, a.L, a.T, tiles_total, nsplit, NW, wid, true);
            if (span.count == 0) return;  // (workgroup-uniform)
            part_slot = (size_t)hk * nsplit * a.B + wid;
            b = span.b;
            bh = b * a.Hkv + hk;
        } else if (tiles_per_wg == 0 && a.B <= 64 && a.B > 2) {
            // rows of one span each: long and short ones are paired on the CUs; outputs stay the batch row's own
            b = __builtin_amdgcn_readfirstlane(balanced_row(a.mask, a.B, a.L, a.T, tiles_total, b));
            bh = b * a.Hkv + hk;
            part_slot = (size_t)bh * nsplit + split;
        }
    }
    const int r = heads_of_a_kv_head<RR>(a.Hq, a.Hkv);
    const int R = r * a.L;  // (a pair's query rows lie one behind the other)

    __shared__ __attribute__((aligned(16))) WaveParts<D, NW, RR> parts;
    // A step with rotary positions: the query rows and the new key row, rotated, wait in LDS (where the partials go at
    // the end) for the wavefronts to fetch them.
    uint16_t *rot_s = reinterpret_cast<uint16_t *>(&parts.rows[0][0][0]);
    [[maybe_unused]] RopeStep<DT, D, NW * 64, 4> step;
    if constexpr (rot)
        step.fetch(a.turn, reinterpret_cast<const uint16_t *>(a.q) + (size_t)bh * R * D,
                   static_cast<const uint16_t *>(a.new_k) + (size_t)bh * D, R);

    // ---- query operands: lane (blk, qi) holds row qi's 4 elements of step 16 x + blk ----
    // qsum[rg][g][i] = sum over group g of the (rounded, fp16-held) query row 4 rg + i, for
    // the bias term; built from the same registers: the 16 steps of one operand pair lie in
    // one group (group sizes of 64 and more; with 32 the lane groups 0-7 and 8-15 feed two sums), so a lane sums its 4 elements, the 16
    // lane groups are added up by shuffles and the four rows are read out of their quad.
    // (Built by a lambda that is called after the first tile has been requested, so the first K/V loads are in flight
    // while the queries are fetched and reduced, and in MODE 3 rotated.)
    Op qa[RG][NQA];
    float qsum[RG][G][4];
    auto load_queries = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        const int i = 4 * rg + qi;
        // rows past R read row 0 (in bounds) and count as zero: no branch around the loads, which
        // are then all in flight together instead of one after the other
        const bool ok = i < R;
        const int row = ok ? i : 0;
        const size_t qoff = ((size_t)bh * R + row) * D;
        float raw[NQA][4];
#pragma unroll
        for (int x = 0; x < NQA; ++x) {
            const int step = 16 * x + blk;
            const int w = step / GEO::WSTEPS, h = step % GEO::WSTEPS;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int d = w * GEO::EPW + GEO::elem(h, k);
                raw[x][k] = rot ? Elem<DT>::load(rot_s, row * D + d) : Elem<DT>::load(a.q, qoff + d);
            }
        }
        float part[G];
#pragma unroll
        for (int g = 0; g < G; ++g) part[g] = 0.f;
#pragma unroll
        for (int x = 0; x < NQA; ++x) {
            float qv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float v = ok ? (float)(_Float16)round_dt<DT>(raw[x][k] * a.scale) : 0.f;
                if constexpr (HALF) {  // steps 16 x + blk: lane groups 0-7 are one group of 32, 8-15 the next
                    part[2 * x] += blk < 8 ? v : 0.f;
                    part[2 * x + 1] += blk < 8 ? 0.f : v;
                } else {
                    part[(64 * x) / GS] += v;
                }
                qv[k] = GEO::hi(k) ? v * 0.0625f : v;
            }
            qa[rg][x].u[0] = pack_h2(qv[0], qv[1]);
            qa[rg][x].u[1] = pack_h2(qv[2], qv[3]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float v = part[g];
            for (int off = 4; off < 64; off <<= 1) v += __shfl_xor(v, off);  // over the 16 lane groups
#pragma unroll
            for (int ii = 0; ii < 4; ++ii)  // wave-uniform: keep it in a scalar register
                qsum[rg][g][ii] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), ii));
        }
    }
    };

    // ---- running state ---------------------------------------------------------------
    // m_use = m_run, or 0 while m_run is still -inf, so exp2((s - m_use) log2 e) needs no guard
    float m_run[RG][4], m_use[RG][4], l_part[RG][4], bacc[RG][G][4];
    f4 oacc[RG][NH];
    f4 oacc2[RG][NO2];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
#pragma unroll
        for (int h = 0; h < NO2; ++h) oacc2[rg][h] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) { m_run[rg][i] = -INFINITY; m_use[rg][i] = 0.f; l_part[rg][i] = 0.f; }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) bacc[rg][g][i] = 0.f;
#pragma unroll
        for (int h = 0; h < NH; ++h) oacc[rg][h] = f4{0.f, 0.f, 0.f, 0.f};
    }

    const float fill = finfo_min_dt(DT);
    [[maybe_unused]] SymMask sym{};
    int tile_begin = split * tiles_per_wg;
    int tile_end = min(tiles_total, tile_begin + tiles_per_wg);
    if constexpr (MM == 1) {
        // length-aware partition: an index-only mask bounds the rows this (batch) can see
        // (left padding, lengths, causal/window reach); spans of equal size start at the first
        // visible tile
        if (__builtin_expect(tiles_per_wg < 0, 0)) {
            sym = span.sym;
            tile_begin = span.t.lo;
            tile_end = span.t.hi;
        } else {
            sym = sym_mask_init(a.mask, b, a.L, a.T);
            const TileRange vis = visible_tiles(sym, tiles_total, true);
            // tiles_per_wg == 0: divide this batch row's own visible range over the spans
            const int per = tiles_per_wg > 0 ? tiles_per_wg
                                             : (max(vis.hi - vis.lo, 1) + nsplit * NW - 1) / (nsplit * NW) * NW;
            tile_begin = vis.lo + split * per;  // spans past the last tile are empty
            tile_end = min(vis.hi, tile_begin + per);
        }
    }
    [[maybe_unused]] KeyBounds seen[RG][4];  // what each carried row sees (formed behind the first requests)
    // tokens whose V code sits in a high nibble carry 1/16 on the probability side
    const float vfac = (BITS == 4 && (lane & 2)) ? 0.0625f : 1.0f;

    constexpr int VROW = T::VW * 4;  // bytes of one V tile row

    // This wavefront takes tiles tile0, tile0 + NW, ...: always the same tile of
    // successive pages (4 tiles each), so its four plane pointers advance by NW / 4 page
    // cell strides.
    const int tile0 = tile_begin + wave;
    const int my_tiles = tile0 < tile_end ? (tile_end - tile0 + NW - 1) / NW : 0;
    constexpr int PSTEP = NW / 4;  // pages per step
    // pages are found through the page table: one scalar load per plane pair and page; the
    // offsets of this (b, kv-head)'s cell and of the tile inside it are the same in every page
    const int tip = tile0 & 3;  // 4 tiles per page
    int page_k = my_tiles > 0 ? tile0 >> 2 : 0, page_v = page_k;
    const size_t k_off = (size_t)bh * st.k_cell + (size_t)tip * TILE * st.k_row;
    const size_t v_off = (size_t)bh * st.v_cell + (size_t)tip * D * VROW;
    const size_t ksb_off = (size_t)bh * st.ksb_cell + (size_t)tip * TILE * st.ksb_row;
    const size_t vsb_off = (size_t)bh * st.vsb_cell + (size_t)tip * TILE * st.vsb_row;
    // Four wavefronts: entries by scalar loads, and the offsets added where the tile's loads are formed, so that nothing
    // waits for an entry before then.  Eight (the chip full of them) read 2 % faster where a half tile's loads arrive
    // before the next are requested, which a page entry that is a vector load of its own sees to: 32768 keys of 256 pairs at
    // 4 bits 196.9 us, 200.7 with scalar entries, 199 with a wait in the loop, 201.5 in workgroups of four.
    constexpr bool LATE = NW == 4;
    using Table = typename std::conditional<LATE, ptab, const PageEntry *>::type;
    const Table pt = (Table) reinterpret_cast<uintptr_t>(st.pt);
    gptr kp = as_global(pt[page_k].k) + (LATE ? 0 : k_off), ksp = as_global(pt[page_k].ksb) + (LATE ? 0 : ksb_off);
    gptr vp = as_global(pt[page_v].v) + (LATE ? 0 : v_off), vsp = as_global(pt[page_v].vsb) + (LATE ? 0 : vsb_off);
    // (the new row's page, if there is one to write: looked up with the first tile's, for one wait)
    const ptab own_page = page_table(st) + (max(a.new_slot, 0) >> PAGE_SHIFT);
    char *const own_pk = own_page->k, *const own_pks = own_page->ksb, *const own_pv = own_page->v, *const own_pvs = own_page->vsb;
    if constexpr (LATE && MM == 0) asm volatile("" ::"s"(own_pk), "s"(own_pks), "s"(own_pv), "s"(own_pvs), "s"(kp), "s"(ksp), "s"(vp), "s"(vsp));
    const uint32_t k_lane = lane * st.k_row, v_lane = lane * VROW;
    const uint32_t ksb_lane = lane * st.ksb_row, vsb_lane = lane * st.vsb_row;
    int slot_next = tile0 * TILE + lane;  // slot of this lane's token in the tile loaded next
    int base_next = tile0 * TILE;         // its first slot (wave-uniform)
    // rows every query row keeps: tiles inside [full_lo, full_hi] need no mask or bound test
    int full_lo = 0, full_hi = a.T - 1;
    if constexpr (MM == 1) {
        sym_mask_full_range(sym, full_lo, full_hi);
        full_hi = min(full_hi, a.T - 1);
    }

    // ---- the step's new row, when it is still to be written (unmasked single-token decode) -----
    // Slot T - 1 lies in the last tile, which exactly one wavefront of one workgroup reads, as its last one (spans
    // are equal and cover every tile).  The wavefronts of that workgroup quantize the row into the cache, with the arithmetic
    // of the append kernel, behind their first tile's request and in front of any other: the row's keys and values go in units
    // of UC columns (whole groups), shared out from the wavefront behind the tile's reader on, which has the most tiles.  A
    // barrier stands between the row and later loads of the row's tile; if that is its reader's first, it is requested only then.
    // V codes go into their columns' packed words read-modify-write; the row and the old words are requested in front of the tile.
    // (The whole row quantized by the tile's reader, the last wavefront of the launch to finish: 16 layers of 512 keys x 64 at 8 bits
    // 109.6 us for 107.6, four of 30 000 x 128 at 4 bits 65.8 for 64.5.  The row written first
    // and the tiles requested behind it: by four round trips to memory later.  The row's
    // own tile requested in front as well and once more behind the row: 8 bits, one sequence of 2000 keys x 64, the step
    // 10.6 us for 10.2; 60 keys x 128 9.5 for 9.2.)
    constexpr int UC = GS > 64 ? GS : 64, EU = UC / 64, NU = D / UC, UPW = (2 * NU + NW - 1) / NW;  // columns and elements of a lane in a unit; units of a side and of a wavefront
    bool row_here = false, own = false;  // workgroup-uniform; wave-uniform: reads the row's tile
    int unit0 = 2 * NU;                  // this wavefront's first unit: 0 .. NU - 1 keys, NU .. 2 NU - 1 values
    uint32_t row_e[UPW][EU], row_w[UPW][EU];
    if constexpr (MM == 0 && RG == 1) {
        if (a.new_k != nullptr) {  // wave-uniform
            const int slot = a.new_slot, tl = slot >> 6;
            row_here = tl >= tile_begin && tl < tile_end;
            if (row_here) {
                const int reader = (tl - tile_begin) % NW;
                own = wave == reader;
                unit0 = (wave - reader - 1 + 2 * NW) % NW;
                const uint16_t *krow = static_cast<const uint16_t *>(a.new_k) + (size_t)bh * D;
                const uint16_t *vrow = static_cast<const uint16_t *>(a.new_v) + (size_t)bh * D;
                const char *vcell = own_pv + (size_t)bh * st.v_cell;
#pragma unroll
                for (int j = 0; j < UPW; ++j) {
                    const int u = unit0 + j * NW;
                    if (u < 2 * NU && !(rot && u < NU)) {
#pragma unroll
                        for (int e = 0; e < EU; ++e) {
                            const int d = (u < NU ? u : u - NU) * UC + 64 * e + lane;
                            if (u < NU) {
                                row_e[j][e] = krow[d];
                            } else {
                                row_e[j][e] = vrow[d];
                                row_w[j][e] = reinterpret_cast<const uint32_t *>(vcell + v_row_off(st, slot, d))[v_bitpos<BITS>(slot & (TILE - 1)) >> 5];
                            }
                        }
                    }
                }
            }
        }
    }
    auto write_row = [&]() __attribute__((always_inline)) {
        const int slot = a.new_slot, bp = v_bitpos<BITS>(slot & (TILE - 1));
        const size_t in_page = slot & (PAGE - 1);
#pragma unroll
        for (int j = 0; j < UPW; ++j) {
            // (the elements' first use, and so the wait for them: turned into floats as soon as they were loaded, they were
            // waited for in front of the first tile's request)
#pragma unroll
            for (int e = 0; e < EU; ++e) asm("" : "+v"(row_e[j][e]));
            const int u = unit0 + j * NW, from = (u < NU ? u : u - NU) * UC;
            if (u < NU) {
                quantize_row_wave_from<DT, BITS>(
                    [&](int d) { return rot ? Elem<DT>::load(rot_s, R * D + d) : pair_scale<DT>(row_e[j][EU == 1 ? 0 : (d - lane - from) >> 6]); }, from + UC, GS, lane,
                    reinterpret_cast<uint32_t *>(own_pk + (size_t)bh * st.k_cell + in_page * st.k_row), [](int, uint32_t) {},
                    own_pks + (size_t)bh * st.ksb_cell + in_page * st.ksb_row, nullptr, nullptr, from);
            } else if (u < 2 * NU) {
                char *vcell = own_pv + (size_t)bh * st.v_cell;
                quantize_row_wave_from<DT, BITS>(
                    [&](int d) { return pair_scale<DT>(row_e[j][EU == 1 ? 0 : (d - lane - from) >> 6]); }, from + UC, GS, lane, nullptr,
                    [&](int d, uint32_t code) {
                        reinterpret_cast<uint32_t *>(vcell + v_row_off(st, slot, d))[bp >> 5] =
                            (row_w[j][EU == 1 ? 0 : (d - lane - from) >> 6] & ~(((1u << BITS) - 1u) << (bp & 31))) | (code << (bp & 31));
                    },
                    own_pvs + (size_t)bh * st.vsb_cell + in_page * st.vsb_row, nullptr, nullptr, from);
            }
        }
    };

    // The K half (codes, scales, row bookkeeping) and the V half of tile number k_loaded /
    // v_loaded of this wavefront (clamped to its last tile, so loads past the end stay
    // unconditional and in bounds).
    int k_loaded = 0, v_loaded = 0;
    auto load_k = [&](T &t) {
        load_words<T::KW>(t.k, kp + (LATE ? k_off : 0) + k_lane);
        load_words<G>(t.ksb, ksp + (LATE ? ksb_off : 0) + ksb_lane);
        t.row = slot_next < a.T ? slot_next : -1;
        t.edge = base_next < full_lo || base_next + (TILE - 1) > full_hi;
        ++k_loaded;
        if (k_loaded < my_tiles) {  // wave-uniform: step to the same tile of the next page
            page_k += PSTEP;
            kp = as_global(pt[page_k].k) + (LATE ? 0 : k_off);
            ksp = as_global(pt[page_k].ksb) + (LATE ? 0 : ksb_off);
            slot_next += PAGE * PSTEP;
            base_next += PAGE * PSTEP;
        }
    };
    auto load_v = [&](T &t) {
#pragma unroll
        for (int h = 0; h < NH; ++h) load_words<T::VW>(t.v[h], vp + (LATE ? v_off : 0) + v_lane + (size_t)h * 64 * VROW);
        load_words<G>(t.vsb, vsp + (LATE ? vsb_off : 0) + vsb_lane);
        ++v_loaded;
        if (v_loaded < my_tiles) {
            page_v += PSTEP;
            vp = as_global(pt[page_v].v) + (LATE ? 0 : v_off);
            vsp = as_global(pt[page_v].vsb) + (LATE ? 0 : vsb_off);
        }
    };
    auto load_tile = [&](T &t) {
        load_k(t);
        load_v(t);
    };

    Op pa[RG][G];  // probabilities of the tile in flight, as PV operands
    auto compute_qk_softmax = [&](const T &t) {
        const bool live = t.row >= 0;
        // ---- QK^T: scores of token `lane` for every query row ---------------------------
        f4 sacc[RG][G];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int g = 0; g < G; ++g) sacc[rg][g] = f4{0.f, 0.f, 0.f, 0.f};
        static_for<T::KW>([&](auto W) {
            constexpr int w = decltype(W)::value;
            constexpr int g = (w * GEO::EPW) / GS;
            Op o[GEO::WSTEPS];
            GEO::unpack(t.k[w], o);
            static_for<GEO::WSTEPS>([&](auto H) {
                constexpr int h = decltype(H)::value;
                constexpr int step = w * GEO::WSTEPS + h;
#pragma unroll
                for (int rg = 0; rg < RG; ++rg)
                    sacc[rg][g] = mfma444<step % 16>(qa[rg][step / 16], o[h], sacc[rg][g]);
            });
        });

        // ---- online softmax per row group; probabilities become PV A operands ------------
        // Interior tiles (every token live and visible to every query row: the common case,
        // decided per wavefront when the tile was loaded) skip all mask and bound tests.
        float ks24[G], vsf[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            ks24[g] = pair_scale<DT>(t.ksb[g]) * TWO24;
            vsf[g] = pair_scale<DT>(t.vsb[g]) * vfac;
        }
        auto softmax_rg = [&](auto RGC) {
            constexpr int rg = decltype(RGC)::value;
            float sc[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float s_ = pair_bias<DT>(t.ksb[0]) * qsum[rg][0][i];
#pragma unroll
                for (int g = 1; g < G; ++g) s_ = __builtin_fmaf(pair_bias<DT>(t.ksb[g]), qsum[rg][g][i], s_);
#pragma unroll
                for (int g = 0; g < G; ++g) s_ = __builtin_fmaf(ks24[g], sacc[rg][g][i], s_);
                sc[i] = round_dt<DT>(s_);
            }
            if (MM == 2 || t.edge) {  // wave-uniform
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float s_ = sc[i];
                    [[maybe_unused]] const int row_i = 4 * rg + i;
                    if constexpr (MM == 1) {
                        if (!seen[rg][i].keep(t.row)) s_ = fill;
                    } else if constexpr (MM == 2) {
                        if (live && row_i < R) {
                            const int rep = row_i / a.L, l = row_i - rep * a.L;
                            float add;
                            const bool keep = mask_keep(a.mask, b, hk * r + rep, l, t.row, a.L, a.T, add);
                            if (!keep) s_ = fill;
                            else if (a.mask.dtype != KVHIP_BOOL) s_ = round_dt<DT>(s_ + add);
                        }
                    }
                    sc[i] = live ? s_ : -INFINITY;
                }
            }
            // raise the running maximum only when this tile exceeds it (rare after the first
            // few tiles; the empty asm keeps the reductions inside the branch)
            bool need = false;
#pragma unroll
            for (int i = 0; i < 4; ++i) need = need || (sc[i] > m_run[rg][i]);
            if (__any(need)) {
                float top[4] = {sc[0], sc[1], sc[2], sc[3]};
                asm volatile("" : "+v"(top[0]));
                wave_max4(top);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // wave-uniform values, kept in scalar registers
                    const float mn = uniform(fmaxf(m_run[rg][i], top[i]));
                    const float alpha = (mn == -INFINITY) ? 1.f : fast_exp2((m_run[rg][i] - mn) * LOG2E);
                    m_run[rg][i] = mn;
                    m_use[rg][i] = uniform((mn == -INFINITY) ? 0.f : mn);
                    l_part[rg][i] *= alpha;
#pragma unroll
                    for (int g = 0; g < G; ++g) bacc[rg][g][i] *= alpha;
#pragma unroll
                    for (int h = 0; h < NH; ++h) oacc[rg][h][i] *= alpha;
                    if constexpr (HALF) {
#pragma unroll
                        for (int h = 0; h < NH; ++h) oacc2[rg][h][i] *= alpha;
                    }
                }
            }
            constexpr int GP = (G + 1) / 2;  // groups travel through the transpose two to a register
            uint32_t x[GP][4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // exp2(-inf) = 0 covers dead lanes; m_use is finite even before any live token
                const float p = fast_exp2((sc[i] - m_use[rg][i]) * LOG2E);
                l_part[rg][i] += p;
                float pv[2 * GP];
                pv[2 * GP - 1] = 0.f;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    bacc[rg][g][i] = __builtin_fmaf(p, pair_bias<DT>(t.vsb[g]), bacc[rg][g][i]);
                    pv[g] = p * vsf[g];
                }
#pragma unroll
                for (int j = 0; j < GP; ++j) x[j][i] = pack_h2(pv[2 * j], pv[2 * j + 1]);
            }
            // lane (blk, i) now gets, in x[j][k], row i's value for token 4 blk + k
#pragma unroll
            for (int j = 0; j < GP; ++j) {
                quad_transpose(x[j], lane);
                pa[rg][2 * j].u[0] = __builtin_amdgcn_perm(x[j][1], x[j][0], 0x05040100u);
                pa[rg][2 * j].u[1] = __builtin_amdgcn_perm(x[j][3], x[j][2], 0x05040100u);
                if (2 * j + 1 < G) {
                    pa[rg][2 * j + 1].u[0] = __builtin_amdgcn_perm(x[j][1], x[j][0], 0x07060302u);
                    pa[rg][2 * j + 1].u[1] = __builtin_amdgcn_perm(x[j][3], x[j][2], 0x07060302u);
                }
            }
        };
        static_for<RG>([&](auto RGC) { softmax_rg(RGC); });
    };

    // ---- out += P . V: lane supplies column lane (+64 h), step s = tokens 4s..4s+3 ----------
    auto compute_pv = [&](const T &t) {
        static_for<NH>([&](auto HH) {
            constexpr int h = decltype(HH)::value;
            constexpr int g = HALF ? 2 * h : (64 * h) / GS;
            static_for<T::VW>([&](auto W) {
                constexpr int w = decltype(W)::value;
                Op o[GEO::WSTEPS];
                GEO::unpack(t.v[h][w], o);
                static_for<GEO::WSTEPS>([&](auto S2) {
                    constexpr int s = w * GEO::WSTEPS + decltype(S2)::value;
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) {
                        oacc[rg][h] = mfma444<s>(pa[rg][g], o[decltype(S2)::value], oacc[rg][h]);
                        if constexpr (HALF)
                            oacc2[rg][h] = mfma444<s>(pa[rg][g + 1], o[decltype(S2)::value], oacc2[rg][h]);
                    }
                });
            });
        });
    };

    auto compute_tile = [&](const T &t) {
        compute_qk_softmax(t);
        compute_pv(t);
    };

    // ---- main loop.  Variants whose tile fits twice in the register file keep one whole
    // tile of loads in flight ahead of the arithmetic.  The others run one buffer with the
    // halves skewed: V of a tile is requested before its QK^T and softmax, K of the next
    // tile before its PV, so each half has the other half's arithmetic to arrive in.
    constexpr bool PREFETCH = (RG == 1 && !(BITS == 8 && D >= 128)) || (BITS == 4 && D <= 128 && (RG == 2 || D == 64));
    T first;
    auto request_first = [&]() __attribute__((always_inline)) {
        if constexpr (PREFETCH) load_tile(first);
        else load_k(first);
    };
    const bool row_first = own && my_tiles == 1;  // wave-uniform: the first tile is the new row's
    if (my_tiles > 0 && !row_first) request_first();
    if constexpr (MM == 1) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int i = 0; i < 4; ++i) seen[rg][i] = sym_mask_bounds(sym, (4 * rg + i) % a.L);
    }
    if constexpr (rot) {
        step.turn(a.turn, bh, R, rot_s);
        __syncthreads();
    }
    if constexpr (MM == 0 && RG == 1) {
        if (row_here) {  // workgroup-uniform
            write_row();
            __syncthreads();
            if (row_first) request_first();
        }
    }
    if (my_tiles > 0) {
        load_queries();
        if constexpr (PREFETCH) {
            T bufB;
            for (int done = 0;;) {
                load_tile(bufB);
                compute_tile(first);
                if (++done == my_tiles) break;
                load_tile(first);
                compute_tile(bufB);
                if (++done == my_tiles) break;
            }
        } else {
            for (int done = 0; done < my_tiles; ++done) {
                load_v(first);
                compute_qk_softmax(first);
                load_k(first);
                compute_pv(first);
            }
        }
    }

    // ---- the wavefronts' parts -> LDS ---------------------------------------------------
    if (lane == 0)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) *reinterpret_cast<f4 *>(&parts.m[wave][4 * rg]) = f4{m_run[rg][0], m_run[rg][1], m_run[rg][2], m_run[rg][3]};
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        wave_sum4(l_part[rg]);
#pragma unroll
        for (int g = 0; g < G; ++g) wave_sum4(bacc[rg][g]);
    }
    __syncthreads();  // (the rotated rows have been fetched, too)
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        float wgt[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) wgt[i] = wave_weight(parts, 4 * rg + i, m_run[rg][i]);
        if (lane == 0) *reinterpret_cast<f4 *>(&parts.l[wave][4 * rg]) = f4{wgt[0] * l_part[rg][0], wgt[1] * l_part[rg][1], wgt[2] * l_part[rg][2], wgt[3] * l_part[rg][3]};
#pragma unroll
        for (int h = 0; h < NH; ++h) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float o_ = oacc[rg][h][i], b_ = bacc[rg][HALF ? 2 * h : (64 * h) / GS][i];
                if constexpr (HALF) {
                    if (lane >= 32) {
                        o_ = oacc2[rg][h][i];
                        b_ = bacc[rg][2 * h + 1][i];
                    }
                }
                parts.rows[wave][4 * rg + i][64 * h + lane] = wgt[i] * (o_ * TWO24 + b_);
            }
        }
    }
    __syncthreads();
    if constexpr (MM == 1) {
        if (tiles_per_wg < 0 && nsplit > 1 && wid == span.first && threadIdx.x == 0)  // (for the merge)
            span_table(a.workspace, st.BH, nsplit, RR * (D + 2))[bh] = make_int2((int)part_slot, span.count);
    }
    // a single span writes the output rows, several leave partials
    leave_rows<D, DT>(a, parts, R, nsplit == 1, (size_t)bh * R, part_slot);
}

// ---------------------------------------------------------------------------------
// Full-precision caches (KVCacheSimple, RotatingKVCache), fp16 or bf16.
//
// Same decomposition and the same 4x4x4 broadcast contraction as above, but a tile of
// 16-bit K and V is 4x larger than a 4-bit one, so it is streamed through two
// 32-register buffers in pieces of 64 elements per lane: a K piece is 64 head-dim
// elements of the lane's token, a V piece is the 64 tokens of the lane's column.
// The load of the next piece is issued as soon as a buffer has been consumed.
// bf16 keeps P as a (hi, lo) pair of bf16 values so the PV product carries 16 bits of
// probability; rows of a RotatingKVCache are found through the run table.
template <int D, int DT, int RG, int MODE, bool IDENT>
__global__ void __launch_bounds__(WAVES * 64, 2)
decode_fp_kernel(int tiles_total, int tiles_per_wg, int nsplit, typename DecodeArgs<MODE>::type a) {
    fetch_arguments(a, tiles_total, tiles_per_wg, nsplit);
    constexpr int MM = MODE == 3 ? 0 : MODE;
    constexpr bool rot = MODE == 3;
    constexpr bool BF = DT == 1;
    constexpr int NP = D / 64;   // pieces per K row and per V tile column set
    constexpr int RR = 4 * RG;
    constexpr int PW = 32;       // dwords per piece
    const Store &st = a.st;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int blk = lane >> 2, qi = lane & 3;
    int bh = blockIdx.y;
    const int split = blockIdx.x;
    int b = MM == 0 ? 0 : bh / a.Hkv;  // (without a mask nothing asks for it)
    [[maybe_unused]] const int hk = bh - b * a.Hkv;
    const int r = heads_of_a_kv_head<RR>(a.Hq, a.Hkv);
    const int R = r * a.L;  // (a pair's query rows lie one behind the other)
    size_t part_slot = (size_t)bh * nsplit + split;  // where this workgroup's partial goes
    [[maybe_unused]] RaggedSpan span;
    [[maybe_unused]] int wid = 0;
    if constexpr (MM == 1 && IDENT) {
        if (__builtin_expect(tiles_per_wg < 0, 0)) {  // a ragged batch that shares its spans out (behind the rest of the kernel)
            wid = b * nsplit + split;
            span = ragged_span(a.mask, a.B, a.L, a.T, tiles_total, nsplit, WAVES, wid, false);
            if (span.count == 0) return;  // (workgroup-uniform)
            part_slot = (size_t)hk * nsplit * a.B + wid;
            b = span.b;
            bh = b * a.Hkv + hk;
        }
    }

    __shared__ __attribute__((aligned(16))) WaveParts<D, WAVES, RR> parts;
    // A step with rotary positions: the query rows and the new key row, rotated, wait in LDS (where the partials go at
    // the end) for the wavefronts to fetch them.
    uint16_t *rot_s = reinterpret_cast<uint16_t *>(&parts.rows[0][0][0]);
    [[maybe_unused]] RopeStep<DT, D, WAVES * 64, RR> step;
    if constexpr (rot)
        step.fetch(a.turn, reinterpret_cast<const uint16_t *>(a.q) + (size_t)bh * R * D,
                   static_cast<const uint16_t *>(a.new_k) + (size_t)bh * D, R);

    // query operands: lane (blk, qi) holds row qi's elements 4*(16 x + blk) .. +3, unscaled
    Op qa[RG][NP];
    auto load_queries = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
            const int i = 4 * rg + qi;
            const size_t qoff = ((size_t)bh * R + i) * D;
#pragma unroll
            for (int x = 0; x < NP; ++x) {
                uint2 w = make_uint2(0, 0);
                if (i < R) {
                    if (rot) w = *reinterpret_cast<const uint2 *>(rot_s + i * D + 4 * (16 * x + blk));
                    else w = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(a.q) + qoff + 4 * (16 * x + blk));
                }
                qa[rg][x].u[0] = w.x;
                qa[rg][x].u[1] = w.y;
            }
        }
    };

    float m_run[RG][4], l_part[RG][4];
    f4 oacc[RG][NP];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
#pragma unroll
        for (int i = 0; i < 4; ++i) { m_run[rg][i] = -INFINITY; l_part[rg][i] = 0.f; }
#pragma unroll
        for (int h = 0; h < NP; ++h) oacc[rg][h] = f4{0.f, 0.f, 0.f, 0.f};
    }

    [[maybe_unused]] SymMask sym{};
    int tile_begin = split * tiles_per_wg;
    int tile_end = min(tiles_total, tile_begin + tiles_per_wg);
    if constexpr (MM == 1 && IDENT) {
        if (__builtin_expect(tiles_per_wg < 0, 0)) {
            sym = span.sym;
            tile_begin = span.t.lo;
            tile_end = span.t.hi;
        } else {
            sym = sym_mask_init(a.mask, b, a.L, a.T);
            const TileRange vis = visible_tiles(sym, tiles_total, false);
            // tiles_per_wg == 0: divide this batch row's own visible range over the spans
            const int per = tiles_per_wg > 0 ? tiles_per_wg
                                             : (max(vis.hi - vis.lo, 1) + nsplit * WAVES - 1) / (nsplit * WAVES) * WAVES;
            tile_begin = vis.lo + split * per;  // spans past the last tile are empty
            tile_end = min(vis.hi, tile_begin + per);
        }
    } else if constexpr (MM == 1) {
        sym = sym_mask_init(a.mask, b, a.L, a.T);
    }
    [[maybe_unused]] KeyBounds seen[RG][4];  // what each carried row sees (formed behind the first requests)
    const int tile0 = tile_begin + wave;
    const int my_tiles = tile0 < tile_end ? (tile_end - tile0 + WAVES - 1) / WAVES : 0;
    // a wavefront's tiles are a page apart: each is found through the page table (a scalar load)
    const int tip = tile0 & 3;
    int page_k = my_tiles > 0 ? tile0 >> 2 : 0, page_v = page_k;
    constexpr int VROW = TILE * 2;  // bytes of one V tile row
    const size_t k_off = (size_t)bh * st.k_cell + (size_t)tip * TILE * st.k_row;
    const size_t v_off = (size_t)bh * st.v_cell + (size_t)tip * D * VROW;
    const ptab pt = page_table(st);
    gptr kp = as_global(pt[page_k].k), vp = as_global(pt[page_v].v);
    // chunk-interleaved tiles: chunk j of the lane's token (K) or column (V) sits 16 * lane bytes into
    // a 1 KB (K) / 16 D byte (V) row of chunks, so every load below is contiguous across the wavefront
    const uint32_t k_lane = lane * 16, v_lane = lane * 16;
    int slot_cur = tile0 * TILE + lane;
    int k_loaded = 0, v_loaded = 0;  // tiles whose K / V pieces have been requested
    auto load_chunks = [&](uint32_t *buf, gptr p, size_t stride) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PW / 4; ++j) {
            const kv_u4 v = ld_global<kv_u4>(p + (size_t)j * stride);
            buf[4 * j] = v.x; buf[4 * j + 1] = v.y; buf[4 * j + 2] = v.z; buf[4 * j + 3] = v.w;
        }
    };

    // piece x of the K row / V column set of the tile the respective pointer stands on;
    // after the last piece the pointer steps to this wavefront's next tile (clamped, so
    // the prefetch past the end stays unconditional and in bounds)
    auto load_k = [&](uint32_t *buf, int x) {
        load_chunks(buf, kp + k_off + k_lane + (size_t)x * (PW / 4) * (TILE * 16), TILE * 16);  // chunks 8x .. 8x+7 of the lane's token
        if (x == NP - 1) {
            ++k_loaded;
            if (k_loaded < my_tiles) kp = as_global(pt[++page_k].k);
        }
    };
    auto load_v = [&](uint32_t *buf, int x) {
        load_chunks(buf, vp + v_off + v_lane + (size_t)x * 64 * 16, (size_t)D * 16);  // the 8 token chunks of column 64x + lane
        if (x == NP - 1) {
            ++v_loaded;
            if (v_loaded < my_tiles) vp = as_global(pt[++page_v].v);
        }
    };

    // piece order per tile: K0 .. K(NP-1), V0 .. V(NP-1); piece n lives in buffer n % NBUF and piece
    // n + NBUF is requested as soon as piece n has been consumed.  Two buffers: four (32 KB per
    // wavefront in flight) measured slower on the short launches they were meant for (a 4096-row
    // sliding window at D = 256, one tile per wavefront: 17.4 us against 15.7 us).
    constexpr int NBUF = KVHIP_DECODE_FP_NBUF(D, RG);
    uint32_t bufs[NBUF][PW];
    auto buf_of = [&](int n) -> uint32_t * { return bufs[n % NBUF]; };
    // request piece n (counted from the start of a tile; past its end: of the next tile) into `buf`
    auto request = [&](uint32_t *buf, int n) __attribute__((always_inline)) {
        n %= 2 * NP;
        if (n < NP) load_k(buf, n);
        else load_v(buf, n - NP);
    };

    // ---- the step's new row, when it is still to be written (unmasked single-token decode) -----
    // Exactly one wavefront of one workgroup reads the tile of physical slot `new_slot` (spans are equal and
    // cover every tile): it copies the row into the page after it has requested its first pieces and before it requests
    // others, so its own later loads of the tile see it; if its first tile is that tile, of the first pieces the K ones are
    // requested ahead all the same and their lane of the row's token is given the row from LDS.  (All of them requested behind
    // the row, with a wait for its stores, that wavefront ended the kernel.)  The row is
    // requested in front of the pieces.
    bool own = false;
    kv_u4 own_k;
    uint32_t own_v[NP];
    if constexpr (MM == 0) {
        if (a.new_k != nullptr) {  // wave-uniform
            const int tl = a.new_slot >> 6;
            own = tl >= tile_begin && tl < tile_end && ((tl - tile_begin) % WAVES) == wave;
            if (own) {
                if constexpr (!rot) {  // one 16-byte chunk of the K row per lane
                    if (lane < D / 8) own_k = ld_global<kv_u4>(as_global(a.new_k) + ((size_t)bh * D + 8 * lane) * 2);
                }
#pragma unroll
                for (int h = 0; h < NP; ++h) own_v[h] = ld_global<uint16_t>(as_global(a.new_v) + ((size_t)bh * D + 64 * h + lane) * 2);
            }
        }
    }
    // (the queries before the pieces: loads complete in order, and a wait for queries requested after the
    // first pieces would be a wait for those pieces too -- in every iteration, the compiler
    // placing one wait for all ways into the loop)
    constexpr int NK = NBUF < NP ? NBUF : NP;  // K pieces among the first
    auto request_first_k = [&]() __attribute__((always_inline)) {
        static_for<NK>([&](auto N) { request(buf_of(decltype(N)::value), decltype(N)::value); });
    };
    auto request_first_v = [&]() __attribute__((always_inline)) {
        static_for<NBUF - NK>([&](auto N) { request(buf_of(NK + decltype(N)::value), NK + decltype(N)::value); });
    };
    const bool row_first = own && tile0 == a.new_slot >> 6;  // wave-uniform
    if (my_tiles > 0) {
        if constexpr (!rot) load_queries();
        request_first_k();
        if (!row_first) request_first_v();
    }
    if constexpr (MM == 1) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int i = 0; i < 4; ++i) seen[rg][i] = sym_mask_bounds(sym, (4 * rg + i) % a.L);
    }
    if constexpr (rot) {
        step.turn(a.turn, bh, R, rot_s);
        __syncthreads();
        if (my_tiles > 0) load_queries();
    }
    if constexpr (MM == 0) {
        if (own) {  // wave-uniform
            // (global stores: behind a store to a plain pointer every load in flight is waited for.  What a
            // wavefront loads behind its own stores it loads as stored: the fence holds the compiler)
            const int slot = a.new_slot, tk = slot & (TILE - 1);
            const PageEntry page{const_cast<char *>(pt[a.new_slot >> PAGE_SHIFT].k), nullptr, const_cast<char *>(pt[a.new_slot >> PAGE_SHIFT].v), nullptr};
            KV_GLOBAL char *kc = (KV_GLOBAL char *)as_global(page.k + (size_t)bh * st.k_cell);
            KV_GLOBAL char *vc = (KV_GLOBAL char *)as_global(page.v + (size_t)bh * st.v_cell);
            uint16_t *row_s = rot ? rot_s + R * D : reinterpret_cast<uint16_t *>(&parts.rows[wave][0][0]);
            if (lane < D / 8) {
                if constexpr (rot) own_k = *reinterpret_cast<const kv_u4 *>(row_s + 8 * lane);
                else *reinterpret_cast<kv_u4 *>(row_s + 8 * lane) = own_k;
                *reinterpret_cast<KV_GLOBAL kv_u4 *>(kc + kfp_at<2>(2 * D, slot, 8 * lane)) = own_k;
            }
#pragma unroll
            for (int h = 0; h < NP; ++h) *reinterpret_cast<KV_GLOBAL uint16_t *>(vc + vfp_at<2>(D, slot, 64 * h + lane)) = (uint16_t)own_v[h];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (row_first) {
                request_first_v();
                if (lane == tk) {
                    static_for<NK>([&](auto X) {
                        constexpr int x = decltype(X)::value;
                        uint32_t *buf = buf_of(x);
#pragma unroll
                        for (int j = 0; j < PW / 4; ++j) {
                            const kv_u4 v = *reinterpret_cast<const kv_u4 *>(row_s + 64 * x + 8 * j);
                            buf[4 * j] = v.x; buf[4 * j + 1] = v.y; buf[4 * j + 2] = v.z; buf[4 * j + 3] = v.w;
                        }
                    });
                }
            }
        }
    }
    if (my_tiles > 0) {
        for (int done = 0; done < my_tiles; ++done) {
            int row;
            if (IDENT) row = slot_cur;
            else row = slot_cur < a.slots ? slot_to_row(a.runs, slot_cur) : -1;
            row = (row >= 0 && row < a.T) ? row : -1;
            const bool live = row >= 0;
            // ---- QK^T over the K pieces ---------------------------------------------
            f4 sacc[RG];
#pragma unroll
            for (int rg = 0; rg < RG; ++rg) sacc[rg] = f4{0.f, 0.f, 0.f, 0.f};
            static_for<NP>([&](auto X) {
                constexpr int x = decltype(X)::value;
                uint32_t *buf = buf_of(x);
                static_for<16>([&](auto S) {
                    constexpr int s = decltype(S)::value;
                    Op o;
                    o.u[0] = buf[2 * s];
                    o.u[1] = buf[2 * s + 1];
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg)
                        sacc[rg] = BF ? mfma444_bf<s>(qa[rg][x], o, sacc[rg]) : mfma444<s>(qa[rg][x], o, sacc[rg]);
                });
                // the buffer is free: request the piece NBUF ahead in the order K.., V.., next tile's K..
                request(buf, x + NBUF);
            });
            // ---- online softmax ----------------------------------------------------------
            Op pa[RG], pl[RG];
#pragma unroll
            for (int rg = 0; rg < RG; ++rg) {
                float sc[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float s_ = sacc[rg][i] * a.scale;
                    [[maybe_unused]] const int row_i = 4 * rg + i;
                    if constexpr (MM == 1) {
                        if (!seen[rg][i].keep(row)) s_ = -INFINITY;
                    } else if constexpr (MM == 2) {
                        if (live && row_i < R) {
                            const int rep = row_i / a.L, l = row_i - rep * a.L;
                            float add;
                            const bool keep = mask_keep(a.mask, b, hk * r + rep, l, row, a.L, a.T, add);
                            s_ = keep ? s_ + add : -INFINITY;
                        }
                    }
                    sc[i] = live ? s_ : -INFINITY;
                }
                bool need = false;
#pragma unroll
                for (int i = 0; i < 4; ++i) need = need || (sc[i] > m_run[rg][i]);
                if (__any(need)) {
                    float top[4] = {sc[0], sc[1], sc[2], sc[3]};
                    asm volatile("" : "+v"(top[0]));  // keeps the reductions inside the branch
                    wave_max4(top);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float mn = fmaxf(m_run[rg][i], top[i]);
                        const float alpha = (mn == -INFINITY) ? 1.f : fast_exp2((m_run[rg][i] - mn) * LOG2E);
                        m_run[rg][i] = mn;
                        l_part[rg][i] *= alpha;
#pragma unroll
                        for (int h = 0; h < NP; ++h) oacc[rg][h][i] *= alpha;
                    }
                }
                uint32_t xx[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = (sc[i] == -INFINITY || m_run[rg][i] == -INFINITY) ? 0.f : fast_exp2((sc[i] - m_run[rg][i]) * LOG2E);
                    l_part[rg][i] += p;
                    if (BF) {
                        const uint32_t hi = Elem<1>::bits(p);
                        const float rest = p - __uint_as_float(hi << 16);
                        xx[i] = hi | ((uint32_t)Elem<1>::bits(rest) << 16);
                    } else {
                        xx[i] = (uint32_t)f2h_bits(p);
                    }
                }
                quad_transpose(xx, lane);
                pa[rg].u[0] = __builtin_amdgcn_perm(xx[1], xx[0], 0x05040100u);
                pa[rg].u[1] = __builtin_amdgcn_perm(xx[3], xx[2], 0x05040100u);
                if (BF) {
                    pl[rg].u[0] = __builtin_amdgcn_perm(xx[1], xx[0], 0x07060302u);
                    pl[rg].u[1] = __builtin_amdgcn_perm(xx[3], xx[2], 0x07060302u);
                }
            }
            // ---- out += P . V over the V pieces ---------------------------------------------
            static_for<NP>([&](auto X) {
                constexpr int x = decltype(X)::value;
                uint32_t *buf = buf_of(NP + x);
                static_for<16>([&](auto S) {
                    constexpr int s = decltype(S)::value;
                    Op o;
                    o.u[0] = buf[2 * s];
                    o.u[1] = buf[2 * s + 1];
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) {
                        if (BF) {
                            oacc[rg][x] = mfma444_bf<s>(pa[rg], o, oacc[rg][x]);
                            oacc[rg][x] = mfma444_bf<s>(pl[rg], o, oacc[rg][x]);
                        } else {
                            oacc[rg][x] = mfma444<s>(pa[rg], o, oacc[rg][x]);
                        }
                    }
                });
                request(buf, NP + x + NBUF);
            });
            slot_cur += PAGE;
        }
    }

    if (lane == 0)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) *reinterpret_cast<f4 *>(&parts.m[wave][4 * rg]) = f4{m_run[rg][0], m_run[rg][1], m_run[rg][2], m_run[rg][3]};
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) wave_sum4(l_part[rg]);
    __syncthreads();  // (the rotated rows have been fetched, too)
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        float wgt[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) wgt[i] = wave_weight(parts, 4 * rg + i, m_run[rg][i]);
        if (lane == 0) *reinterpret_cast<f4 *>(&parts.l[wave][4 * rg]) = f4{wgt[0] * l_part[rg][0], wgt[1] * l_part[rg][1], wgt[2] * l_part[rg][2], wgt[3] * l_part[rg][3]};
#pragma unroll
        for (int h = 0; h < NP; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) parts.rows[wave][4 * rg + i][64 * h + lane] = wgt[i] * oacc[rg][h][i];
    }
    __syncthreads();
    if constexpr (MM == 1 && IDENT) {
        if (tiles_per_wg < 0 && nsplit > 1 && wid == span.first && threadIdx.x == 0)  // (for the merge)
            span_table(a.workspace, st.BH, nsplit, RR * (D + 2))[bh] = make_int2((int)part_slot, span.count);
    }
    // a single span writes the output rows itself, several leave partials for the merge kernel
    leave_rows<D, DT>(a, parts, R, nsplit == 1, (size_t)bh * R, part_slot);
}

struct Plan {
    int tiles_total, tiles_per_wg, nsplit, rg, nw;
};

// Quantized shapes that run on the 16-row kernel at every row count: head size 96 (a row and a half of the 4-row
// kernel's 64-column halves), keys of 192 with values of 128, and 2-, 3-, 5- and 6-bit codes (bit streams, which
// the 4-row kernel's whole-word operands do not read).
static bool only_decode16(const Store &s) {
    return s.bits != 0 && (s.Dk == 96 || s.Dk == 192 || (s.bits != 4 && s.bits != 8));
}

Plan plan_for(const AttendArgs &a) {
    Plan p;
    p.tiles_total = (a.slots + TILE - 1) / TILE;
    const int R = (a.Hq / a.Hkv) * a.L;
    p.rg = R <= 4 ? 1 : (R <= 8 ? 2 : 4);
    const int BH = a.st.BH;
    // Spans are sized so that all workgroups are resident at once (2 per CU): every
    // wavefront streams for the whole kernel and no second scheduling round leaves CUs
    // idle.  A span is a multiple of WAVES tiles so each wavefront gets the same share.
    // (the full-precision kernel, whose tiles are 4x larger, measured faster with one
    // workgroup per CU: 46 us against 52 us at 8192 tokens, B8, 8 kv heads, D 128)
    int want = (a.st.bits != 0 ? 256 * 2 : 256) / BH;
    if (want < 1) want = 1;
    int per = (p.tiles_total + want - 1) / want;
    // KVHIP_DECODE_TILES forces the span size in tiles (timing builds only: measure_knob)
    static const int forced_tiles = measure_knob("KVHIP_DECODE_TILES", 0);
    if (forced_tiles > 0) per = forced_tiles;
    // short sequences (up to 1024 quantized or 512 full-precision rows): one span per pair, so the
    // kernel writes the output rows itself and the merge launch, which costs more than the split
    // gains at this size, is not needed (B1, 4 kv heads, 640 rows, 8-bit: 19.5 -> 16.8 us per step)
    else if (p.tiles_total <= (a.st.bits != 0 ? 4 * WAVES : 2 * WAVES)) per = p.tiles_total;
    per = per < WAVES ? WAVES : per;
    per = (per + WAVES - 1) / WAVES * WAVES;
    while ((p.tiles_total + per - 1) / per > 512) per *= 2;  // the merge kernel holds 512 span weights
    p.tiles_per_wg = per;
    p.nsplit = (p.tiles_total + per - 1) / per;
    // ragged batches (per-batch bounds), marked by tiles_per_wg < 0: up to 64 rows share the launch's workgroups out by
    // their lengths (ragged_span); 0: more rows, or one span each, where every row divides its own visible range
    // over the same number of spans.  Both need slots in presented order: a
    // ring presented through a row map keeps equal spans over all of its slots.
    p.nw = WAVES;
    const bool ident = a.runs.n == 1 && a.runs.row0[0] == 0 && a.runs.phys0[0] == 0;
    if (a.mask.mode == KVHIP_MASK_WINDOW && (a.mask.left_pad || a.mask.lengths) && forced_tiles <= 0 && ident) {
        const bool paired = a.st.bits != 0 && a.B > 2;  // (balanced_row, in the quantized kernels)
        p.tiles_per_wg = a.B >= 2 && a.B <= 64 && p.nsplit >= (paired ? 3 : 2) && p.tiles_total > p.nsplit * WAVES ? -1 : 0;
        // KVHIP_RAGGED_SPANS forces the number of spans per batch row (timing builds only: measure_knob)
        static const int forced_spans = measure_knob("KVHIP_RAGGED_SPANS", 0);
        if (forced_spans > 0) p.nsplit = std::min(forced_spans, 512);
    } else if (a.st.bits != 0 && p.nsplit >= 2 && want <= 4 && p.rg == 1 && !only_decode16(a.st) && a.mask.mode != KVHIP_MASK_ARRAY &&
               forced_tiles <= 0) {
        // 128 pairs or more: workgroups of 8 wavefronts, one per CU -- the same wavefronts per CU
        // with half the spans.  With 256 pairs a workgroup takes its pair's whole sequence: the
        // merge stays on chip and the kernel writes the output itself (no partials, no second
        // launch).  Measured at 32k tokens, 4-bit, D 128: B32 207 -> 204 us, B16 112 -> 107 us.
        p.nw = 2 * WAVES;
        int w8 = 256 / BH;
        if (w8 < 1) w8 = 1;
        int per8 = (p.tiles_total + w8 - 1) / w8;
        per8 = (per8 + p.nw - 1) / p.nw * p.nw;
        p.tiles_per_wg = per8;
        p.nsplit = (p.tiles_total + per8 - 1) / per8;
    }
    // a caller with a fixed amount of scratch: fewer, longer spans until the partials fit (one span has none)
    if (a.workspace_cap) {
        const size_t per_span = (size_t)BH * (a.st.bits != 0 && (p.rg >= 2 || only_decode16(a.st)) ? 16 : 4 * p.rg) *
                                (a.st.Dv + 2) * sizeof(float);
        while (p.nsplit > 1 && per_span * p.nsplit + BH * sizeof(int2) > a.workspace_cap) {
            if (p.tiles_per_wg > 0) {
                p.tiles_per_wg *= 2;
                p.nsplit = (p.tiles_total + p.tiles_per_wg - 1) / p.tiles_per_wg;
            } else {
                p.nsplit /= 2;
            }
        }
        if (p.nsplit == 1) p.tiles_per_wg = std::max(p.tiles_per_wg, 0);
    }
    return p;
}

// (per calling thread: a thread brackets and reads its own launches)
thread_local int g_profile = 0;        // 0 off, n: bracket every n-th launch of the dominant kernel
thread_local int g_profile_count = 0;  // launches seen since it was enabled
thread_local bool g_profile_open = false;
thread_local std::vector<hipEvent_t> g_events;  // begin/end pairs

}  // namespace

void profile_enable(int every) {
    g_profile = every > 0 ? every : 0;
    g_profile_count = 0;
    g_profile_open = false;
}

void profile_mark(hipStream_t s, bool begin) {
    if (!g_profile) return;
    if (begin) {
        g_profile_open = (g_profile_count++ % g_profile) == 0;
        if (!g_profile_open) return;
    } else if (!g_profile_open) {
        return;
    }
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return;
    (void)hipEventRecord(e, s);
    g_events.push_back(e);
}

hipError_t profile_read(int *launches, double *total_ms) {
    *launches = 0;
    *total_ms = 0.0;
    for (size_t i = 0; i + 1 < g_events.size(); i += 2) {
        hipError_t e = hipEventSynchronize(g_events[i + 1]);
        if (e != hipSuccess) return e;
        float ms = 0.f;
        e = hipEventElapsedTime(&ms, g_events[i], g_events[i + 1]);
        if (e != hipSuccess) return e;
        *total_ms += ms;
        *launches += 1;
    }
    for (hipEvent_t ev : g_events) (void)hipEventDestroy(ev);
    g_events.clear();
    return hipSuccess;
}

bool attend_decode_supported(const AttendArgs &a) {
    const Store &s = a.st;
    if (s.dtype != KVHIP_F16 && s.dtype != KVHIP_BF16) return false;
    // keys of 192 with values of 128 (the multi-head latent attention models): quantized caches, on the 16-row kernel
    const bool mla = s.Dk == 192 && s.Dv == 128 && s.bits != 0;
    if (s.Dk != s.Dv && !mla) return false;
    const int R = (a.Hq / a.Hkv) * a.L;
    if (R > 16) return false;
    // full precision: more than 8 rows (4 at D = 256) are faster on the prefill tile than on further
    // passes of the broadcast contraction (8192 keys, 8 kv heads: B16 D 128 16 rows 104 us against
    // 164 us; B8 D 256 8 rows about 105 us against 133 us)
    if (s.bits == 0) return (s.Dk == 64 || s.Dk == 128 || s.Dk == 256) && R <= (s.Dk == 256 ? 4 : 8);
    if (a.runs.n != 1 || a.runs.row0[0] != 0 || a.runs.phys0[0] != 0) return false;
    if (s.bits != 4 && s.bits != 8) return decode16_stream_shape(s);  // every row count on the 16-row kernel
    if (s.Dk == 64) return s.gs == 32 || s.gs == 64;
    if (s.Dk == 96) return s.gs == 32;  // every row count on the 16-row kernel
    if (mla) return s.gs == 32 || s.gs == 64;  // likewise
    if (s.Dk == 128) return s.gs == 32 || s.gs == 64 || s.gs == 128;
    if (s.Dk == 256) return s.gs == 64 || s.gs == 128;
    return false;
}

// The decode kernels -- the 4-row and the 16-row quantized kernel and the full-precision one --, without a mask, write
// a single-token step's new row themselves.
bool attend_decode_fuses_append(const AttendArgs &a) {
    if (!attend_decode_supported(a) || a.L != 1 || a.mask.mode != KVHIP_MASK_NONE) return false;
    static const bool off = measure_knob("KVHIP_NO_FUSED_APPEND", 0) != 0;  // (timing builds only)
    return !off;
}

// 5..16 rows per kv head of a quantized cache go to the 16x16x32 kernel
// (kvhip_attend_decode16.hip), which always carries 16 rows: measured faster than the 4-row
// broadcast contraction from 8 rows up (B16, 8 kv heads, 8192 tokens: 37 us against 43 us at
// 8 rows, 36 us against 87 us at 16).
// The shapes of only_decode16() take it for every row count.
static bool use_decode16(const AttendArgs &a, const Plan &p) {
    return a.st.bits != 0 && (p.rg >= 2 || only_decode16(a.st));
}

size_t attend_decode_workspace(const AttendArgs &a) {
    const Plan p = plan_for(a);
    const int rows = use_decode16(a, p) ? 16 : 4 * p.rg;
    if (p.nsplit == 1) return 0;  // a single span writes the output rows itself: no partials
    return (size_t)a.st.BH * p.nsplit * rows * (a.st.Dv + 2) * sizeof(float)  // (partials hold output columns)
           + (p.tiles_per_wg < 0 ? a.st.BH * sizeof(int2) : 0);
}

hipError_t launch_attend_decode(const AttendArgs &a_in, hipStream_t s) {
    const AttendArgs &a = a_in;
    const Plan p = plan_for(a);
    const Store &st = a.st;
    dim3 grid(p.nsplit, st.BH), block(WAVES * 64);  // the quantized kernel sets its own block size
    const int mm = decode_mode(a);
    auto spans_of = [&](int rows) { return p.tiles_per_wg < 0 ? span_table(a.workspace, st.BH, p.nsplit, rows * (st.Dv + 2)) : nullptr; };
#define DEC_K(BITS, D, GS, DT, RG, MM, NW)                                                                \
    hipLaunchKernelGGL((decode_kernel<BITS, D, GS, DT, RG, MM, NW>), grid, dim3(NW * 64), 0, s, p.tiles_total, p.tiles_per_wg, \
                       p.nsplit, DecodeArgs<MM>::type(a))
#define DEC(BITS, D, GS, DT, RG)                                                                          \
    do {                                                                                                  \
        profile_mark(s, true);                                                                            \
        if (p.nw == 2 * WAVES) {                                                                          \
            if (mm == 0) DEC_K(BITS, D, GS, DT, RG, 0, 2 * WAVES);                                        \
            else if (mm == 3) DEC_K(BITS, D, GS, DT, RG, 3, 2 * WAVES);                                   \
            else DEC_K(BITS, D, GS, DT, RG, 1, 2 * WAVES);                                                \
        } else if (mm == 0) {                                                                             \
            DEC_K(BITS, D, GS, DT, RG, 0, WAVES);                                                         \
        } else if (mm == 3) {                                                                             \
            DEC_K(BITS, D, GS, DT, RG, 3, WAVES);                                                         \
        } else if (mm == 1) {                                                                             \
            DEC_K(BITS, D, GS, DT, RG, 1, WAVES);                                                         \
        } else {                                                                                          \
            DEC_K(BITS, D, GS, DT, RG, 2, WAVES);                                                         \
        }                                                                                                 \
        profile_mark(s, false);                                                                           \
        if (p.nsplit > 1)                                                                                 \
            (void)launch_combine(a, p.nsplit, 4 * RG, s, spans_of(4 * RG));                              \
    } while (0)
#define DEC_RG(BITS, D, GS, DT) DEC(BITS, D, GS, DT, 1) /* more rows: the 16-row kernel above */
    if (use_decode16(a_in, p)) {
        profile_mark(s, true);
        hipError_t e = launch_attend_decode16(a_in, p.tiles_total, p.tiles_per_wg, p.nsplit, s);
        profile_mark(s, false);
        if (e != hipSuccess) return e;
        if (p.nsplit > 1) return launch_combine(a_in, p.nsplit, 16, s, spans_of(16));
        return hipSuccess;
    }
#define DEC_DT(BITS, D, GS)                                \
    do {                                                   \
        if (st.dtype == KVHIP_F16) DEC_RG(BITS, D, GS, 0); \
        else DEC_RG(BITS, D, GS, 1);                       \
    } while (0)
#define DEC_Q(BITS)                                 \
    do {                                            \
        if (st.Dk == 64 && st.gs == 32) DEC_DT(BITS, 64, 32);   \
        else if (st.Dk == 128 && st.gs == 32) DEC_DT(BITS, 128, 32); \
        else if (st.Dk == 64) DEC_DT(BITS, 64, 64); \
        else if (st.Dk == 256 && st.gs == 64) DEC_DT(BITS, 256, 64);  \
        else if (st.Dk == 256) DEC_DT(BITS, 256, 128);                \
        else if (st.gs == 64) DEC_DT(BITS, 128, 64); \
        else DEC_DT(BITS, 128, 128);                \
    } while (0)
    const bool ident = a.runs.n == 1 && a.runs.row0[0] == 0 && a.runs.phys0[0] == 0;
#define FP(D, DT, RG, M, I)                                                                               \
    do {                                                                                                  \
        profile_mark(s, true);                                                                            \
        hipLaunchKernelGGL((decode_fp_kernel<D, DT, RG, M, I>), grid, block, 0, s, p.tiles_total, p.tiles_per_wg, \
                           p.nsplit, DecodeArgs<M>::type(a));                                                     \
        profile_mark(s, false);                                                                           \
        if (p.nsplit > 1)                                                                                 \
            (void)launch_combine(a, p.nsplit, 4 * RG, s, spans_of(4 * RG));                              \
    } while (0)
#define FP_MI(D, DT, RG)                                          \
    do {                                                          \
        if (mm == 0 && ident) FP(D, DT, RG, 0, true);             \
        else if (mm == 0) FP(D, DT, RG, 0, false);                \
        else if (mm == 3 && ident) FP(D, DT, RG, 3, true);        \
        else if (mm == 3) FP(D, DT, RG, 3, false);                \
        else if (mm == 1 && ident) FP(D, DT, RG, 1, true);        \
        else if (mm == 1) FP(D, DT, RG, 1, false);                \
        else if (ident) FP(D, DT, RG, 2, true);                   \
        else FP(D, DT, RG, 2, false);                             \
    } while (0)
    // (up to 8 query rows per kv head, 4 at D = 256: attend_decode_supported() sends more to the prefill tile)
#define FP_RG(D, DT)                                           \
    do {                                                       \
        if (p.rg == 1) FP_MI(D, DT, 1);                        \
        else if (p.rg == 2 && D < 256) FP_MI(D, DT, (D < 256 ? 2 : 1)); \
        else return hipErrorInvalidValue;                      \
    } while (0)
#define FP_DT(D)                                  \
    do {                                          \
        if (st.dtype == KVHIP_F16) FP_RG(D, 0);   \
        else FP_RG(D, 1);                         \
    } while (0)
    if (st.bits == 4) DEC_Q(4);
    else if (st.bits == 8) DEC_Q(8);
    else if (st.Dk == 64) FP_DT(64);
    else if (st.Dk == 128) FP_DT(128);
    else FP_DT(256);
#undef FP_DT
#undef FP_RG
#undef FP_MI
#undef FP
#undef DEC_Q
#undef DEC_DT
#undef DEC_RG
#undef DEC
#undef DEC_K
    return hipGetLastError();
}

}  // namespace kvhip
