// Chunked-prefill attention for full-precision caches (fp16 / bf16) on the matrix cores
// (gfx950, v_mfma_f32_16x16x32_f16 / _bf16).
//
// One workgroup (4 wavefronts) owns 64 query rows of one (batch, kv-head) pair (grids of few rows, head size 256, keys of
// 192 with values of 128; more rows of head sizes up to 128: kvhip_attend_prefill_rows32.hip) and walks the cached keys in tiles of 32 slots:
//   S^T   = K . Q^T      A = K rows from LDS in the cache's own dtype (no conversion),
//                        B = query rows held in registers
//   out^T += V^T . P^T   A = V^T rows from LDS in the cache's own dtype, B = the probabilities, rounded
//                        to it, exactly where the S^T accumulators left them, so P never moves between lanes
// K/V tiles are double-buffered in LDS and arrive there straight from global memory, K two tiles ahead of its use
// and V one, with a single barrier per tile.  The interleaved page is made of the 16-byte chunks that the operands
// want, so a buffer is the tile's chunks in page order, and its operand reads are bank-conflict free.
// The online softmax rescales the accumulators only when a row maximum rises, and key tiles
// that every query row of the workgroup sees completely skip all mask tests.
#include "kvhip_prefill_fp.hpp"

#ifndef KVHIP_PREFILL_LM
#define KVHIP_PREFILL_LM 1
#endif
// how far ahead of their use the matrix-core operands are read from LDS
#ifndef KVHIP_PF_VG
#define KVHIP_PF_VG 2
#endif
#ifndef KVHIP_PF_NVB
#define KVHIP_PF_NVB 2
#endif
#ifndef KVHIP_PF_AHEAD
#define KVHIP_PF_AHEAD 2
#endif

#ifndef KV_SB
#define KV_SB __builtin_amdgcn_sched_barrier(0)
#endif
namespace kvhip {

namespace {

using namespace prefill_fp;

__device__ __forceinline__ uint32_t rn_h2(float lo, float hi) { return pk_h2(lo, hi); }    // round to nearest even
__device__ __forceinline__ uint32_t rn_bf2(float lo, float hi) { return pk_bf2(lo, hi); }
// c += a . b and c = a . b on the matrix cores.  DT: 0 fp16 operands, 1 bf16 operands.
template <int DT> __device__ __forceinline__ void mfma_acc(f4 &c, const Op8 &a, const Op8 &b) {
    if constexpr (DT == 0) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, b.h, c, 0, 0, 0);
    else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, b.b, c, 0, 0, 0);
}
template <int DT> __device__ __forceinline__ void mfma_new(f4 &c, const Op8 &a, const Op8 &b) {
    c = f4{0.f, 0.f, 0.f, 0.f};
    mfma_acc<DT>(c, a, b);
}
// 16 query rows per wavefront.  (32 at D = 256 need the accumulator registers of
// a whole SIMD lane, one wavefront per SIMD, which measured slower: 0.34 ms against 0.29 ms
// for a 512 x 4607 chunk at B4, 8 query heads.)
//
// The loop is software-pipelined over the key tiles: iteration t issues S^T(t+1) = K(t+1) Q^T on
// the matrix cores and, between those instructions, the vector-ALU half of the softmax of tile t
// (scale, exp2, rounding to 16 bits), whose scores iteration t-1 left in registers; then
// out^T += V(t)^T P(t)^T; then the mask, the tile maximum and the (rare) raise of the reference
// maximum for tile t+1.  One wavefront so keeps the matrix cores and the vector ALU busy at the
// same time, which the in-order issue of a tile-at-a-time loop (scores -> softmax -> PV, each
// waiting for the one before) cannot.  K is requested two tiles ahead and V one tile ahead, each
// into the buffer of its tile's parity; one barrier per iteration.
// DK and DV are the head sizes of keys / queries and of values / outputs (192 and 128 for the multi-head
// latent attention models, equal otherwise).
template <int DK, int DV, int DT, bool IDENT, int MM>
__global__ void __launch_bounds__(256, 2)
prefill_fp_kernel(AttendArgs a, int nsplit) {
    constexpr int BM = 64;
    constexpr int S = (DK + 31) / 32;  // contraction steps over the head dim (the last one partly zero at D = 80)
    constexpr int NDT = DV / 16;   // 16-row tiles of out^T
    constexpr int NCK = (DK + 63) / 64, NCV = (DV + 63) / 64;  // rounds of 256 16-byte chunks, for K and for V
    constexpr int CHK = 4 * DK, CHV = 4 * DV;  // 16-byte chunks of a tile's K and of its V; multiples of 64
    static_assert(DK % 16 == 0 && DV % 16 == 0, "out^T is built from 16-row tiles");
    // A head size that is not a multiple of 32 (80): the last contraction step reads K chunks past the
    // row -- the unused tail that the repeated loads fill with finite values -- against query
    // operands that are zero there.
    static_assert(4 * S * BN <= NCK * 256, "the padded contraction stays inside the staged buffer");
    // K and V tiles move from global memory straight into LDS (no registers, no LDS store
    // instructions): per parity of the tile one buffer for K, the tile's 16-byte chunks in page order
    // [8-element chunk][token], and one for V, [8-token chunk][column].  bf16 caches keep K and V as
    // bf16: the probabilities are rounded to bf16 for the PV matrix-core instruction (the reference's
    // softmax output is an array of the cache's dtype as well).
    // 16-bit elements reserved for a tile's K (and for its V): whole rounds of 256 chunks.  With a head
    // size that is not a multiple of 64 (80, 96) the last round is partly empty: its wavefronts past the
    // tile's last chunk repeat that chunk into the unused tail, so that every wavefront issues the same
    // number of loads.
    constexpr int KSZ = NCK * 256 * 8, VSZ = NCV * 256 * 8;
    __shared__ __attribute__((aligned(16))) uint16_t KV0[KSZ + VSZ], KV1[KSZ + VSZ];
    auto Ks = [&](int par) __attribute__((always_inline)) -> uint16_t * { return par == 0 ? KV0 : KV1; };
    auto Vs = [&](int par) __attribute__((always_inline)) -> uint16_t * { return (par == 0 ? KV0 : KV1) + KSZ; };
    __shared__ int rows_s[2][BN];
    __shared__ int full_s[2];
    __shared__ VisitShared visit_s;

    const Store &st = a.st;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, jj = lane >> 4;
    const int r = a.Hq / a.Hkv;
    const int R = r * a.L;
    const WorkItem item = work_item<MM>(a, (R + BM - 1) / BM, nsplit);
    const int blk_x = item.block, bh = item.bh;
    const int b = MM == 0 ? 0 : bh / a.Hkv;  // (without a mask nothing asks for it)
    [[maybe_unused]] const int hk = bh - b * a.Hkv;
    const int row = blk_x * BM + wave * 16 + n;  // this lane's query row
    const SymMask sym = sym_mask_init(a.mask, b, a.L, a.T);
    // Scores enter the softmax as exp2(s * ef - m) with ef = |scale| log2 e > 0 -- a negative scale
    // flips the sign of the query operands instead (exact), a zero one becomes a vanishing positive
    // factor -- so that the maximum can be taken on the raw scores and the scale folds into one
    // multiply-add.  Under an array mask the mask step leaves s * ef (+ the additive term) in the
    // score registers and the factor is 1.
    // fp16 caches up to D = 128: the denominators ride on the matrix cores (lacc = ones . P^T sums the
    // same rounded probabilities the numerator uses; all 16 rows of the block hold the same sums).
    // D = 256 has no registers to spare, and bf16 keeps float32 denominators.
    constexpr bool LM = DK <= 128 && DV <= 128 && DT == 0 && KVHIP_PREFILL_LM;
    const bool flip = a.scale < 0.f;
    const float sl2 = fmaxf(fabsf(a.scale) * LOG2E, 1e-30f);
    const float ef = MM == 2 ? 1.f : sl2;

    // ---- query operands: B of S^T = K . Q^T; lane (n, jj) holds q[row][32 s + 8 jj ..] raw ----
    Op8 qop[S];
    const bool q_ok = row < R;
    int q_l = 0, q_h = 0;
    {
        // (a pair's query rows lie one behind the other; which positions they are is worked out behind the first requests)
        const u4 *qp = reinterpret_cast<const u4 *>(reinterpret_cast<const uint16_t *>(a.q) + ((size_t)bh * R + row) * DK + 8 * jj);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            qop[s].v = (q_ok && (DK % 32 == 0 || 32 * s + 8 * jj < DK)) ? qp[4 * s] : u4{0, 0, 0, 0};
        }
    }

    f4 oacc[NDT];
    float m_run = -INFINITY, l_run = 0.f;
    [[maybe_unused]] f4 lacc = f4{0.f, 0.f, 0.f, 0.f};
    Op8 ones;
    ones.v = u4{0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u};
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) oacc[dt] = f4{0.f, 0.f, 0.f, 0.f};

    // ---- key tiles this workgroup has to visit, and the rows all of its queries keep ---------
    const Visit visit = visit_plan<BM, MM, IDENT>(a, sym, blk_x, R, item.split, nsplit, visit_s);
    const int keep_lo = visit.keep_lo, keep_hi = visit.keep_hi;
    auto vt_of = [&](int v) __attribute__((always_inline)) -> int { return visit.tile(v); };
    const int v_lo = visit.lo, v_hi = visit.hi;

    // ---- requests -------------------------------------------------------------------------
    // direct global -> LDS: lane i of a wavefront's load lands at the wavefront's LDS base + 16 i, so
    // chunk c = e * 256 + tid goes to slot c of the buffer.  K slot (chunk cc, position pos) takes
    // token 8 ((pos & 15) / 4) + 4 (pos / 16) + pos % 4, the order in which the S^T accumulators of one
    // lane cover the eight tokens of one V chunk (so K operand reads are contiguous across lanes and P
    // never moves), and V slots are the page's own order.
    // A tile of 32 slots inside its page cell (16-bit elements): the 64-token tile t64 starts at
    // t64 * 64 * DK * 2 bytes in the K plane and t64 * 64 * DV * 2 in the V plane; its K chunk (cc, token) lies at
    // (cc * 64 + token) * 16, its V chunk (8-token chunk tc, column) at (tc * DV + column) * 16.
    const size_t cell_k = (size_t)bh * st.k_cell, cell_v = (size_t)bh * st.v_cell;
    PageCursor page_k(st, min(vt_of(v_lo) * BN, max(a.slots - 1, 0))), page_v = page_k;
    // the lane's byte offsets inside a tile, one per round of 256 chunks
    uint32_t koff[NCK], voff[NCV];
#pragma unroll
    for (int e = 0; e < NCK; ++e) {
        const int c = min(e * 256 + tid, CHK - 1);
        const int pos = c % BN;
        const int tok = 8 * ((pos & 15) >> 2) + 4 * (pos >> 4) + (pos & 3);
        koff[e] = (uint32_t)((c / BN) * (TILE * 16) + tok * 16);
    }
#pragma unroll
    for (int e = 0; e < NCV; ++e) voff[e] = (uint32_t)(min(e * 256 + tid, CHV - 1) * 16);
    auto dma_k = [&](int tile, int par) __attribute__((always_inline)) {
        const int slot0 = tile * BN;
        if (wave == (tile & 3) && lane < BN) {  // the wavefronts take this in turn
            const int pos = lane;
            const int slot = slot0 + 8 * ((pos & 15) >> 2) + 4 * (pos >> 4) + (pos & 3);
            int key;
            if (IDENT) key = slot;
            else key = slot < a.slots ? slot_to_row(a.runs, slot) : -1;
            key = (key >= 0 && key < a.T) ? key : -1;
            rows_s[par][pos] = key;  // the row of the token in K slot `pos`
            const bool full = __all(key >= keep_lo && key <= keep_hi);  // (the 32 active lanes)
            if (lane == 0) full_s[par] = full;
        }
        const int t = slot0 & (PAGE - 1);
        const char *kbase = page_k.at(st, slot0).k + cell_k + (size_t)(t >> 6) * (TILE * DK * 2) + (t & 63) * 16;
#pragma unroll
        for (int e = 0; e < NCK; ++e) {
            // whole rounds differ by a constant, which goes to the scalar base; a partly empty last
            // round (its tail repeats the tile's last chunk) keeps its own lane offsets
            if (DK % 64 == 0) load_to_lds(kbase + e * 8 * (TILE * 16), koff[0], &Ks(par)[(e * 256 + 64 * wave) * 8]);
            else load_to_lds(kbase, koff[e], &Ks(par)[(e * 256 + 64 * wave) * 8]);
        }
    };
    auto dma_v = [&](int tile, int par) __attribute__((always_inline)) {
        const int slot0 = tile * BN;
        const int t = slot0 & (PAGE - 1);
        const char *vbase = page_v.at(st, slot0).v + cell_v + (size_t)(t >> 6) * (TILE * DV * 2) + ((t & 63) >> 3) * (DV * 16);
#pragma unroll
        for (int e = 0; e < NCV; ++e) {
            if (DV % 64 == 0) load_to_lds(vbase + e * 256 * 16, voff[0], &Vs(par)[(e * 256 + 64 * wave) * 8]);
            else load_to_lds(vbase, voff[e], &Vs(par)[(e * 256 + 64 * wave) * 8]);
        }
    };
    auto wait_all_loads = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

    // ---- S^T = K . Q^T of one tile: acc[mt] rows = tokens 16 mt + 4 jj + i, column = query n -----
    // operand reads: K slot (chunk 4 s + jj, position 16 mt + n)
    auto read_k = [&](int par, int s, Op8 (&ka)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
            ka[mt].v = *reinterpret_cast<const u4 *>(&Ks(par)[((4 * s + jj) * BN + 16 * mt + n) * 8]);
    };

    // ---- mask of a tile whose scores are in `sc` (raw): excluded keys become -inf; under an array
    // mask the scores are scaled here and additive terms added -----------------------------------
    // An index-only mask (causal, window, per-batch lengths and left padding) keeps, for one query, an
    // interval of key rows: [q_lo, q_lo + q_span] for the query of this lane (empty for a query row
    // past the end), tested with one unsigned comparison per key.
    [[maybe_unused]] int q_lo = 0;
    [[maybe_unused]] uint32_t q_span = 0;
    auto apply_mask = [&](int par, f4 (&sc)[2]) __attribute__((always_inline)) {
        int trow[2][4];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) trow[mt][i] = rows_s[par][16 * mt + 4 * jj + i];  // by K slot; -1: no row
        if constexpr (MM != 2) {
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    bool keep;
                    if constexpr (MM == 1) keep = (uint32_t)(trow[mt][i] - q_lo) <= q_span;
                    else keep = trow[mt][i] >= 0 && q_ok;
                    sc[mt][i] = keep ? sc[mt][i] : -INFINITY;
                }
        } else {
            // a boolean array mask is read four keys at a time where this lane's four rows are consecutive
            bool vec_ok[2];
            uint32_t mword[2] = {0u, 0u};
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
                vec_ok[mt] = a.mask.dtype == KVHIP_BOOL && trow[mt][0] >= 0 && trow[mt][3] == trow[mt][0] + 3 &&
                             trow[mt][1] == trow[mt][0] + 1 && trow[mt][2] == trow[mt][0] + 2;
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
                if (vec_ok[mt] && q_ok) {
                    uint32_t w[1];
                    mask_bool_words<1>(a.mask, b, q_h, q_l, trow[mt][0], w);
                    mword[mt] = w[0];
                }
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float x_ = sc[mt][i] * sl2;
                    const int key = trow[mt][i];
                    bool keep = key >= 0 && q_ok;
                    if (keep) {
                        if (vec_ok[mt]) {
                            keep = ((mword[mt] >> (8 * i)) & 0xffu) != 0u;
                        } else {
                            float add;
                            keep = mask_keep(a.mask, b, q_h, q_l, key, a.L, a.T, add);
                            x_ += add * LOG2E;
                        }
                    }
                    sc[mt][i] = keep ? x_ : -INFINITY;
                }
        }
    };

    // ---- tile maximum and the reference maximum ---------------------------------------------
    // Scores stay in the log2 domain: x = s * ef, p = exp2(x - m).  m is a reference value rather than
    // the exact running maximum: it is the same in the four lanes that share a query and is raised (to
    // the maximum seen) only when a score exceeds it by more than RAISE, so p stays below 2^RAISE
    // (exact in fp16, whose relative precision does not depend on magnitude) and the accumulators are
    // rescaled a handful of times per query, not on every tile that happens to hold a new maximum.
    auto raise = [&](float tmax) __attribute__((always_inline)) {
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        const float mn = fmaxf(m_run, tmax);
        const float alpha = (mn == -INFINITY) ? 1.f : exp2_fast(m_run - mn);
        m_run = mn;
        if constexpr (LM) {
#pragma unroll
            for (int i = 0; i < 4; ++i) lacc[i] *= alpha;
        } else {
            l_run *= alpha;
        }
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) oacc[dt][i] *= alpha;
    };
    auto tile_max = [&](const f4 (&sc)[2]) __attribute__((always_inline)) -> float {
        return ef * fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                          fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
    };
    // The same maximum in four instructions, for the end of an iteration.  `fmaxf` on values the compiler has not
    // seen an arithmetic instruction produce (matrix-core results, selects) first quiets each operand with a
    // maximum of its own: eleven instructions for eight values, on the path every wavefront runs before the
    // barrier.  Written as assembly, which the compiler's hazard handling does not look into: the caller keeps it
    // behind a scheduling barrier that follows the out^T matrix-core instructions, so the score registers, written
    // by matrix-core instructions a whole block earlier (or by the mask's selects), are long complete.
    auto tile_max_raw = [&](const f4 (&sc)[2]) __attribute__((always_inline)) -> float {
        float m;  // (one statement per instruction: the result may then share a register with a finished operand)
        asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(sc[0][0]), "v"(sc[0][1]), "v"(sc[0][2]));
        asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(m), "v"(sc[0][3]), "v"(sc[1][0]));
        asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(m), "v"(sc[1][1]), "v"(sc[1][2]));
        asm volatile("v_max_f32 %0, %1, %2" : "=v"(m) : "v"(m), "v"(sc[1][3]));
        return ef * m;
    };
    // whether the tile whose scores are in `sc` exceeds some query's reference maximum by more than
    // RAISE (wavefront-uniform; a handful of times per query)
    auto needs_raise = [&](const f4 (&sc)[2]) __attribute__((always_inline)) -> bool {
        return __any(tile_max_raw(sc) > m_run + RAISE);
    };
    auto do_raise = [&](const f4 (&sc)[2]) __attribute__((always_inline)) {
        const float tmax = tile_max(sc);
        if (__any(tmax > m_run + RAISE)) raise(tmax);
    };

    // ---- one iteration: tile `tile` (parity PAR) has its scores in `sc`; `sn` receives tile + 1's ---
    // (MASKED: tile + 1 needs its mask evaluated -- a variant of the whole iteration rather than a
    // branch inside it, so that the scores have one definition per variant and the paths join
    // without register copies)
    // The iteration itself never touches the reference maxima or rescales the accumulators: it only
    // reports (`need`) that tile + 1 calls for it, and the loop below leaves its fast part to do so.
    // With the rescaling inside the fast loop the compiler joined the rescaled and the untouched
    // accumulators through register copies on the path that does not rescale: 36 moves per tile at two
    // blocks of 16 query rows, and spills.
    auto body = [&](auto HAS_NEXT_, auto PAR_, auto MASKED_, int tile, f4 (&sc)[2], f4 (&sn)[2], bool &need) __attribute__((always_inline)) {
        constexpr bool HAS_NEXT = decltype(HAS_NEXT_)::value;
        constexpr int PAR = decltype(PAR_)::value;
        constexpr bool MASKED = decltype(MASKED_)::value;
        // the buffers requested into were last read in the previous iteration, which ended with a barrier
        if (tile + 2 < v_hi) dma_k(vt_of(tile + 2), PAR);  // (`tile`: the position in the visiting order)
        if constexpr (HAS_NEXT) dma_v(vt_of(tile + 1), PAR ^ 1);

        float pr[2][4];
        Op8 pb;
        const float negmu = (m_run == -INFINITY) ? 0.f : -m_run;
        // probability `idx` of this lane: accumulator idx
        // (the rounding of a pair of probabilities to 16 bits trails their exp2 by two probabilities, so
        // that it does not wait for a result just asked for)
        auto round_pair = [&](int idx) __attribute__((always_inline)) {  // idx: the odd member of the pair
            const int mt = idx >> 2, i = idx & 3;
            const float p0 = pr[mt][i - 1], p1 = pr[mt][i];
            if constexpr (!LM) l_run += p0 + p1;
            pb.v[2 * mt + (i >> 1)] = DT == 1 ? rn_bf2(p0, p1) : rn_h2(p0, p1);
        };
        constexpr int NP = 8;  // probabilities per lane and tile
        auto softmax_slice = [&](int idx) __attribute__((always_inline)) {
            const int mt = idx >> 2, i = idx & 3;
            pr[mt][i] = exp2_fast(__builtin_fmaf(sc[mt][i], ef, negmu));  // exp2(-inf) = 0 for excluded keys
            if ((idx & 1) && idx >= 3) round_pair(idx - 2);
            if (idx == NP - 1) round_pair(idx);
        };
        // V operands (16 columns each) are read in groups of VG, NVB - 1 groups ahead of their use
        constexpr int VG = KVHIP_PF_VG;
        constexpr int NVB = KVHIP_PF_NVB;
        constexpr int NG = (NDT + VG - 1) / VG;
        Op8 va[NVB][VG];
        auto read_v = [&](int g, Op8 (&dst)[VG]) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < VG; ++x)
                if (VG * g + x < NDT)  // tokens 8 jj .. 8 jj + 7 of column 16 (VG g + x) + n: one chunk
                    dst[x].v = *reinterpret_cast<const u4 *>(&Vs(PAR)[(jj * DV + 16 * (VG * g + x) + n) * 8]);
        };
        if constexpr (HAS_NEXT) {
            constexpr int NM = 2 * S;  // matrix-core instructions of the next tile's scores
            // K operands are asked for AHEAD contraction steps ahead, V's first group near the end
            constexpr int AHEAD = KVHIP_PF_AHEAD;
            constexpr int KA = S < AHEAD + 1 ? S : AHEAD + 1;
            Op8 ka[KA][2];
#pragma unroll
            for (int s = 0; s < (S < AHEAD ? S : AHEAD); ++s) read_k(PAR ^ 1, s, ka[s % KA]);
            KV_SB;
#pragma unroll
            for (int k = 0; k < NM; ++k) {
                // two independent accumulator chains, taken in turn
                const int s = k / 2, mt = k & 1;
                if (mt == 0 && s + AHEAD < S) read_k(PAR ^ 1, s + AHEAD, ka[(s + AHEAD) % KA]);
                if (k == NM - 2) {
#pragma unroll
                    for (int g = 0; g < NVB - 1 && g < NG; ++g) read_v(g, va[g]);
                }
                if (s == 0) mfma_new<DT>(sn[mt], ka[s % KA][mt], qop[s]);
                else mfma_acc<DT>(sn[mt], ka[s % KA][mt], qop[s]);
#pragma unroll
                for (int idx = k * NP / NM; idx < (k + 1) * NP / NM; ++idx) softmax_slice(idx);
                KV_SB;
            }
        } else {
#pragma unroll
            for (int g = 0; g < NVB - 1 && g < NG; ++g) read_v(g, va[g]);
#pragma unroll
            for (int idx = 0; idx < NP; ++idx) softmax_slice(idx);
        }

        // ---- out^T += V^T . P^T: A = V^T chunks from LDS, B = the probabilities where they are ----
        if constexpr (LM) mfma_acc<0>(lacc, ones, pb);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (g + NVB - 1 < NG) read_v(g + NVB - 1, va[(g + NVB - 1) % NVB]);
#pragma unroll
            for (int x = 0; x < VG; ++x)
                if (VG * g + x < NDT) mfma_acc<DT>(oacc[VG * g + x], va[g % NVB][x], pb);
        }

        need = false;
        if constexpr (HAS_NEXT) {
            if constexpr (MASKED) apply_mask(PAR ^ 1, sn);
            KV_SB;  // (tile_max_raw: not before the matrix-core instructions above)
            need = needs_raise(sn);
        }
        // What was requested at the top has to land before the barrier: it has had the whole
        // iteration for it, so the wait is short, and no LDS read of the next iteration meets a load
        // in flight into its buffer.  A plain barrier instead of __syncthreads(): nothing but LDS
        // traffic (drained here) has to be ordered across it.
        wait_all_loads();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    if (v_lo < v_hi) {
        dma_k(vt_of(v_lo), 0);
        dma_v(vt_of(v_lo), 0);
        if (v_lo + 1 < v_hi) dma_k(vt_of(v_lo + 1), 1);
    }
    // (behind the requests: a sign flipped as the queries are loaded put a wait for them in front of the first keys' request)
    if (flip) {
#pragma unroll
        for (int s = 0; s < S; ++s) qop[s].v ^= u4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
    }
    if constexpr (MM != 0) {
        const int rep = q_ok ? row / a.L : 0;
        q_l = q_ok ? row - rep * a.L : 0;
        q_h = hk * r + rep;
    }
    if constexpr (MM == 1) {
        int lo, hi;
        if (sym.mode == KVHIP_MASK_CAUSAL) {
            lo = 0;
            hi = a.T - a.L + q_l;
        } else {
            const int li = sym.offset + q_l;
            lo = sym.pad_b;
            hi = min(li, sym.len_b - 1);
            if (sym.window > 0) lo = max(lo, li - sym.window + 1);
        }
        lo = max(lo, 0);
        hi = min(hi, a.T - 1);
        const bool any = q_ok && hi >= lo;
        q_lo = any ? lo : 0x40000000;  // (none: no row reaches it, row - q_lo wraps to a huge unsigned value)
        q_span = any ? (uint32_t)(hi - lo) : 0u;
    }
    wait_all_loads();
    // (the same wait once more in a form the compiler's bookkeeping sees: it then knows that the
    // query operands have arrived, and does not wait for them -- and with them for every load just
    // issued -- inside the loop)
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), others untouched
    __syncthreads();
    if (v_lo < v_hi) {
        f4 sa[2], sb[2];
        {  // scores of the first tile
#pragma unroll
            for (int s = 0; s < S; ++s) {
                Op8 ka[2];
                read_k(0, s, ka);
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) {
                    if (s == 0) mfma_new<DT>(sa[mt], ka[mt], qop[s]);
                    else mfma_acc<DT>(sa[mt], ka[mt], qop[s]);
                }
            }
            if (MM == 2 || full_s[0] == 0) apply_mask(0, sa);
            do_raise(sa);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // K buffer 0 is free again
        using T_ = std::true_type;
        using F_ = std::false_type;
        using P0 = std::integral_constant<int, 0>;
        using P1 = std::integral_constant<int, 1>;
        int tile = v_lo;  // position in the visiting order
        // one iteration with the variant chosen at run time; false after the last tile
        auto iterate = [&](auto PAR_, f4 (&sc)[2], f4 (&sn)[2], bool &need) __attribute__((always_inline)) -> bool {
            constexpr int PAR = decltype(PAR_)::value;
            const bool has_next = tile + 1 < v_hi;
            // whether tile + 1 needs its mask evaluated (workgroup-uniform): with slots in presented
            // order a comparison of its ends with the rows every query keeps, else the flag its
            // request left in LDS -- asked for before the requests below are formed, which hide its latency
            bool masked = true;
            if constexpr (MM != 2) {
                if constexpr (IDENT) masked = !(vt_of(tile + 1) * BN >= keep_lo && vt_of(tile + 1) * BN + (BN - 1) <= keep_hi);
                else masked = full_s[PAR ^ 1] == 0;
            }
            if (has_next) {
                if (__builtin_amdgcn_readfirstlane(masked)) body(T_{}, PAR_, T_{}, tile, sc, sn, need);
                else if constexpr (MM != 2) body(T_{}, PAR_, F_{}, tile, sc, sn, need);
                ++tile;
                return true;
            }
            body(F_{}, PAR_, F_{}, tile, sc, sn, need);
            return false;
        };
        for (;;) {
            // the fast loop: two iterations (one per buffer parity) per round, left when a tile's scores
            // call for a higher reference maximum -- after an even number of iterations (`odd` false:
            // the next tile's scores are in sa) or an odd one (in sb)
            bool more = true, need = false, odd = false;
            for (;;) {
                more = iterate(P0{}, sa, sb, need);
                odd = true;
                if (!more || need) break;
                more = iterate(P1{}, sb, sa, need);
                odd = false;
                if (!more || need) break;
            }
            if (!more) break;
            if (odd) {  // back to an even count through one iteration outside the fast loop
                do_raise(sb);
                more = iterate(P1{}, sb, sa, need);
                if (!more) break;
                if (need) do_raise(sa);
            } else {
                do_raise(sa);
            }
        }
    }

    // ---- normalise and store: lane (n, jj) holds out[q = n][d = 16 dt + 4 jj + i] ------------
    float l = l_run;
    if constexpr (LM) {
        l = lacc[0];
    } else {
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
    }
    if (!q_ok) return;
    if (nsplit > 1) {
        float *part = a.workspace + (((size_t)bh * nsplit + item.split) * R + row) * (DV + 2);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<kv_part4 *>(part + 16 * dt + 4 * jj) = oacc[dt];
        if (jj == 0) {
            part[DV] = m_run * 0.6931471805599453f;  // back from the log2 domain
            part[DV + 1] = l;
        }
        return;
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    uint16_t *op = reinterpret_cast<uint16_t *>(a.out) + ((size_t)bh * R + row) * DV;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
        const float o0 = oacc[dt][0] * inv, o1 = oacc[dt][1] * inv;
        const float o2 = oacc[dt][2] * inv, o3 = oacc[dt][3] * inv;
        *reinterpret_cast<kv_out4 *>(op + 16 * dt + 4 * jj) = DT == 0 ? kv_out4{rn_h2(o0, o1), rn_h2(o2, o3)} : kv_out4{rn_bf2(o0, o1), rn_bf2(o2, o3)};
    }
}

}  // namespace

hipError_t launch_attend_prefill_fp(const AttendArgs &a, int nsplit, hipStream_t s) {
    const Store &st = a.st;
    const int R = (a.Hq / a.Hkv) * a.L;
    const int bm = 64;
    dim3 grid((unsigned)((R + bm - 1) / bm) * st.BH * nsplit), block(256);  // linear: the kernel maps ids to tiles
    const bool ident = a.runs.n == 1 && a.runs.row0[0] == 0 && a.runs.phys0[0] == 0;
    const int mm = a.mask.mode == KVHIP_MASK_NONE ? 0 : (a.mask.mode == KVHIP_MASK_ARRAY ? 2 : 1);
#define PF_M(DK, DV, DT, MM)                                                                                              \
    do {                                                                                                                  \
        if (ident) hipLaunchKernelGGL((prefill_fp_kernel<DK, DV, DT, true, MM>), grid, block, 0, s, a, nsplit);          \
        else hipLaunchKernelGGL((prefill_fp_kernel<DK, DV, DT, false, MM>), grid, block, 0, s, a, nsplit);               \
    } while (0)
#define PF(DK, DV, DT)                        \
    do {                                      \
        if (mm == 0) PF_M(DK, DV, DT, 0);     \
        else if (mm == 1) PF_M(DK, DV, DT, 1); \
        else PF_M(DK, DV, DT, 2);             \
    } while (0)
#define PF_DT(DK, DV)                              \
    do {                                           \
        if (st.dtype == KVHIP_F16) PF(DK, DV, 0);  \
        else PF(DK, DV, 1);                        \
    } while (0)
    if (st.Dk == 192 && st.Dv == 128) PF_DT(192, 128);  // (multi-head latent attention)
    else if (st.Dk == 64) PF_DT(64, 64);
    else if (st.Dk == 80) PF_DT(80, 80);
    else if (st.Dk == 96) PF_DT(96, 96);
    else if (st.Dk == 128) PF_DT(128, 128);
    else PF_DT(256, 256);
#undef PF_DT
#undef PF
#undef PF_M
    return hipGetLastError();
}

}  // namespace kvhip
