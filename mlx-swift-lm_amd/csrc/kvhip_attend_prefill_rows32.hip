// Chunked-prefill attention for full-precision caches of head sizes up to 128 (fp16 / bf16), 32 query rows per wavefront on
// the matrix cores (gfx950, v_mfma_f32_32x32x16).
//
// Four wavefronts own 128 query rows of one (batch, kv-head) pair and walk the cached keys in blocks of 32 slots:
//   S^T   = K . Q^T      A = K rows from LDS, B = query rows held in registers
//   out^T += V^T . P^T   A = V^T rows from LDS, B = the probabilities where the S^T accumulators left them
// A lane's scores belong to one query (two lanes share one), so a block's softmax is 16 multiply-adds, exponentials and
// eight roundings, its maximum eight instructions, and a block of 32 keys 145 instructions beside 16 matrix-core ones that
// each do twice the work of the 16-row kernel's (that one: 245 beside 34).  Two blocks to an iteration: one barrier, one
// set of requests.
//
// Pipeline: step k issues the scores of block k + 1 and spreads the softmax of block k, whose scores step k - 1 left in
// registers, over those instructions and the first half of out^T's (over the scores' alone: 2 % slower).  K and V
// move from global memory straight into two LDS rings of four blocks, an iteration ahead.  Outputs and partials leave through LDS.
//
// What bounds it: the matrix cores at the clock that the chip's power leaves (timed in turn with parts taken out, 2048 x 8192 is 7 %
// faster without exponentials and 16 % without requests; a large matrix product reaches 1190 TFLOP/s), and for short chunks what
// stands around the loop: of 512 new rows over 2048 keys 3.8 us to the first scores, 2 for the partials and up to 3 for
// the blocks that see fewer keys than the last, of 25.
// Events around the launch (bench.py --workload prefill, D 128, 32q/8kv, causal, TFLOP/s of two runs; before it 32 rows on 16x16x32
// instructions, in turn on one box): bfloat16 2048 x 8192 853-866 -> 952-954, 512 x 8192 717-730 -> 732-745, 4096 x 4096 648-655 -> 773;
// float16 2048 x 8192 857-872 -> 926-931, 512 x 8192 701-708 -> 721-738, and for 512 rows a merge of half the bytes.
#include "kvhip_prefill_fp.hpp"

#ifndef KV_SB
#define KV_SB __builtin_amdgcn_sched_barrier(0)
#endif
namespace kvhip {

namespace {

using namespace prefill_fp;
typedef float f16v __attribute__((ext_vector_type(16)));

template <int DT> __device__ __forceinline__ void mfma32(f16v &c, const Op8 &a, const Op8 &b) {
    if constexpr (DT == 0) c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.h, b.h, c, 0, 0, 0);
    else c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
}

template <int D, int DT, bool IDENT, int MM, int HV>
__global__ void __launch_bounds__(256 * HV, 2)
prefill_rows32_kernel(AttendArgs a, int nsplit) {
    constexpr int BM = 128;
    constexpr int KS = D / 16;           // contraction steps of S^T
    constexpr int NCB = (D + 31) / 32;   // 32-column blocks of out^T (the last one half empty at D = 80)
    constexpr int NL = D / 16;           // 1 KB loads of a block's K, and of its V
    constexpr int BLK = BN * D;          // 16-bit elements of a block's K, and of its V
    static_assert(D % 16 == 0, "whole contraction steps");
    constexpr int KSZ = 4 * BLK, VSZ = 4 * BLK + (D % 32 ? 16 * 8 : 0);  // the rings
    __shared__ __attribute__((aligned(16))) uint16_t ring_s[HV * (KSZ + VSZ)];
    __shared__ int rows_all[HV][IDENT ? 1 : 4][BN];
    __shared__ int full_all[HV][4];
    __shared__ VisitShared visit_s;

    const Store &st = a.st;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave8 & 3, half = HV == 2 ? wave8 >> 2 : 0;  // (rows; which half of the keys)
    const int n = lane & 31, hh = lane >> 5;
    uint16_t *const Ks = ring_s + half * (KSZ + VSZ), *const Vs = Ks + KSZ;
    int (&rows_s)[IDENT ? 1 : 4][BN] = rows_all[half];
    int (&full_s)[4] = full_all[half];
    const int r = a.Hq / a.Hkv;
    const int R = r * a.L;
    const WorkItem item = work_item<MM>(a, (R + BM - 1) / BM, nsplit);
    const int blk_x = item.block, bh = item.bh;
    const int b = MM == 0 ? 0 : bh / a.Hkv;  // (without a mask nothing asks for it)
    [[maybe_unused]] const int hk = bh - b * a.Hkv;
    const SymMask sym = sym_mask_init(a.mask, b, a.L, a.T);
    constexpr bool LM = DT == 0;
    const bool flip = a.scale < 0.f;
    const float sl2 = fmaxf(fabsf(a.scale) * LOG2E, 1e-30f);
    const float ef = MM == 2 ? 1.f : sl2;

    // Query operands, B of S^T = K . Q^T: lane (n, hh) holds q[row][16 s + 8 hh ..] raw.  (A pair's query rows lie one behind
    // the other.  Requested first, they arrive last: 64 rows a load.  Which positions they are is worked out behind the first
    // requests for keys.)
    const int row = blk_x * BM + wave * 32 + n;
    const bool q_ok = row < R;
    int q_l = 0, q_h = 0;
    Op8 qop[KS];
    {
        const u4 *qp = reinterpret_cast<const u4 *>(reinterpret_cast<const uint16_t *>(a.q) + ((size_t)bh * R + row) * D + 8 * hh);
#pragma unroll
        for (int s = 0; s < KS; ++s) qop[s].v = q_ok ? qp[2 * s] : u4{0, 0, 0, 0};
    }
    // float16: the denominators ride on the matrix cores, which sum the rounded probabilities that the numerator uses.
    // Read as the operand of a 16x16x32 instruction the probabilities' lanes are 16 queries by four groups of eight
    // tokens, groups 0 and 2 of queries 0 to 15 and groups 1 and 3 of queries 16 to 31: against ones in the even (odd)
    // groups of the even (odd) rows, lacc's even registers are query lane % 16's sum and the odd ones query 16 + lane % 16's.
    f16v oacc[NCB];
    f4 lacc = f4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
    for (int c = 0; c < NCB; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[c][i] = 0.f;
    Op8 ones;
    {
        const uint32_t one = ((lane >> 4) & 1) == (lane & 1) ? 0x3c003c00u : 0u;
        ones.v = u4{one, one, one, one};
    }
    const bool upper = (lane & 16) != 0;  // this lane's query is one of 16 to 31

    // ---- key tiles this workgroup has to visit, and the rows all of its queries keep ---------
    const Visit visit = visit_plan<BM, MM, IDENT>(a, sym, blk_x, R, item.split, nsplit, visit_s);
    const int keep_lo = visit.keep_lo, keep_hi = visit.keep_hi;
    auto vt_of = [&](int v) __attribute__((always_inline)) -> int { return visit.tile(v); };
    int v_lo = visit.lo;
    const int v_hi = visit.hi;
    // two groups of four wavefronts take half of the blocks each; both pass the same barriers
    const int nb_all = max(v_hi - v_lo, 0), nb_first = HV == 2 ? (nb_all + 1) >> 1 : nb_all;
    if (half) v_lo += nb_first;
    const int nb = half ? nb_all - nb_first : nb_all > 0 ? nb_first : 0;
    const int idle = HV == 2 ? (max(nb_first, 1) + 1) / 2 - (max(nb, 1) + 1) / 2 : 0;  // iterations that the other group has more

    // ---- requests ----
    const size_t cell_k = (size_t)bh * st.k_cell, cell_v = (size_t)bh * st.v_cell;
    PageCursor page_k(st, min(vt_of(v_lo) * BN, max(a.slots - 1, 0))), page_v = page_k;
    // position p of a block's K takes token 16 (p / 16) + 8 ((p / 4) & 1) + 4 ((p / 8) & 1) + p % 4
    const uint32_t koff = (uint32_t)(hh * (TILE * 16) + (16 * (n >> 4) + 8 * ((n >> 2) & 1) + 4 * ((n >> 3) & 1) + (n & 3)) * 16);
    const uint32_t voff = (uint32_t)(lane * 16);
    auto request_k = [&](int k, int slot) __attribute__((always_inline)) {  // block k of the visiting order
        const int blk = vt_of(v_lo + min(k, nb - 1)), slot0 = blk * BN;
        if constexpr (!IDENT) {
            if (wave == (k & 3) && lane < BN) {
                const int s_ = slot0 + lane;
                int rw = s_ < a.slots ? slot_to_row(a.runs, s_) : -1;
                rw = (rw >= 0 && rw < a.T) ? rw : -1;
                rows_s[slot][lane] = rw;
                const bool full = __all(rw >= keep_lo && rw <= keep_hi);
                if (lane == 0) full_s[slot] = full;
            }
        }
        const int t = slot0 & (PAGE - 1);
        const char *base = page_k.at(st, slot0).k + cell_k + (size_t)(t >> 6) * (TILE * D * 2) + (t & 63) * 16;
#pragma unroll
        for (int e = 0; e < (NL + 3) / 4; ++e)
            if (4 * e + 3 < NL || 4 * e + wave < NL)
                load_to_lds(base + (4 * e + wave) * (2 * TILE * 16), koff, &Ks[slot * BLK + (4 * e + wave) * 512]);
    };
    auto request_v = [&](int k, int slot) __attribute__((always_inline)) {
        const int blk = vt_of(v_lo + min(k, nb - 1)), slot0 = blk * BN;
        const int t = slot0 & (PAGE - 1);
        const char *base = page_v.at(st, slot0).v + cell_v + (size_t)(t >> 6) * (TILE * D * 2) + ((t & 63) >> 3) * (D * 16);
#pragma unroll
        for (int e = 0; e < (NL + 3) / 4; ++e)
            if (4 * e + 3 < NL || 4 * e + wave < NL)
                load_to_lds(base + (4 * e + wave) * 1024, voff, &Vs[slot * BLK + (4 * e + wave) * 512]);
    };

    // ---- masks ----
    [[maybe_unused]] int q_lo = 0;
    [[maybe_unused]] uint32_t q_span = 0;
    auto masked_block = [&](int k, int slot) __attribute__((always_inline)) -> bool {
        if constexpr (MM == 2) return true;
        if constexpr (IDENT) {
            const int r0 = vt_of(v_lo + k) * BN;
            return !(r0 >= keep_lo && r0 + (BN - 1) <= keep_hi);
        }
        return full_s[slot] == 0;
    };
    // score register 4 (2 t + u) + j of a lane is token 16 t + 8 hh + 4 u + j of the block
    auto apply_mask = [&](int k, int slot, f16v &sc) __attribute__((always_inline)) {
        const int r0 = IDENT ? vt_of(v_lo + k) * BN : 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            int trow[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int tok = 16 * (g >> 1) + 8 * hh + 4 * (g & 1) + j;
                if constexpr (IDENT) trow[j] = (MM == 1 || r0 + tok < a.T) ? r0 + tok : -1;
                else trow[j] = rows_s[IDENT ? 0 : slot][tok];
            }
            if constexpr (MM != 2) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    bool keep;
                    if constexpr (MM == 1) keep = (uint32_t)(trow[j] - q_lo) <= q_span;
                    else keep = trow[j] >= 0 && q_ok;
                    sc[4 * g + j] = keep ? sc[4 * g + j] : -INFINITY;
                }
            } else {
                const bool vec = a.mask.dtype == KVHIP_BOOL && trow[0] >= 0 && trow[3] == trow[0] + 3 && trow[1] == trow[0] + 1 && trow[2] == trow[0] + 2;
                uint32_t w[1] = {0u};
                if (vec && q_ok) mask_bool_words<1>(a.mask, b, q_h, q_l, trow[0], w);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float x = sc[4 * g + j] * sl2;
                    bool keep = trow[j] >= 0 && q_ok;
                    if (keep) {
                        if (vec) {
                            keep = ((w[0] >> (8 * j)) & 0xffu) != 0u;
                        } else {
                            float add;
                            keep = mask_keep(a.mask, b, q_h, q_l, trow[j], a.L, a.T, add);
                            x += add * LOG2E;
                        }
                    }
                    sc[4 * g + j] = keep ? x : -INFINITY;
                }
            }
        }
    };
    // The reference maximum of a query is raised only when a score exceeds it by more than RAISE (in log2 units), so
    // probabilities stay below 2^RAISE and the accumulators are rescaled a handful of times.
    auto do_raise = [&](const f16v &sc) __attribute__((always_inline)) {
        float t = sc[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) t = fmaxf(t, sc[i]);
        t *= ef;
        if (!__any(t > m_run + RAISE)) return;
        t = fmaxf(t, __shfl_xor(t, 32));
        const float mn = fmaxf(m_run, t);
        const float alpha = (mn == -INFINITY) ? 1.f : exp2_fast(m_run - mn);
        m_run = mn;
        if constexpr (LM) {
            const float across = __shfl_xor(alpha, 16), even = upper ? across : alpha, odd = upper ? alpha : across;
            lacc *= f4{even, odd, even, odd};
        } else {
            l_run *= alpha;
        }
#pragma unroll
        for (int c = 0; c < NCB; ++c) oacc[c] *= alpha;
    };

    // ---- one block ----
    const uint16_t *kl = Ks + (hh * BN + n) * 8, *vl = Vs + (hh * D + n) * 8;  // this lane's operand reads
    constexpr int KA = 3, VA = 3, AH = 2;
    // the softmax of a block is spread over the matrix-core instructions of the next scores and the first half of its own
    // output's, which need the first half of the probabilities
    constexpr int SLOTS = KS + NCB;
    auto step = [&](const f16v &sc, f16v &sn, int slot, bool &need) __attribute__((always_inline)) {
        const uint16_t *kp = kl + slot * BLK, *vp = vl + slot * BLK;
        Op8 ka[KA], va[VA], pb[2];
        auto read_k = [&](int s) __attribute__((always_inline)) { ka[s % KA].v = *reinterpret_cast<const u4 *>(kp + 2 * s * BN * 8); };
        auto read_v = [&](int x) __attribute__((always_inline)) {
            va[x % VA].v = *reinterpret_cast<const u4 *>(vp + (2 * (x / NCB) * D + 32 * (x % NCB)) * 8);
        };
        const float negm = (m_run == -INFINITY) ? 0.f : -m_run;
        float pr[16];
        auto round_pair = [&](int i) __attribute__((always_inline)) {  // i: the odd member
            if constexpr (!LM) l_run += pr[i - 1] + pr[i];
            pb[i >> 3].v[(i >> 1) & 3] = DT == 1 ? pk_bf2(pr[i - 1], pr[i]) : pk_h2(pr[i - 1], pr[i]);
        };
        auto prob = [&](int i) __attribute__((always_inline)) {
            pr[i] = exp2_fast(__builtin_fmaf(sc[i], ef, negm));
            if ((i & 1) && i >= 3) round_pair(i - 2);
            if (i == 15) round_pair(15);
        };
#pragma unroll
        for (int s = 0; s < AH && s < KS; ++s) read_k(s);
        KV_SB;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (s + AH < KS) read_k(s + AH);
            else if (s + AH - KS < 2 * NCB) read_v(s + AH - KS);
            if (s == 0) {
                f16v z;
#pragma unroll
                for (int i = 0; i < 16; ++i) z[i] = 0.f;
                sn = z;
            }
            mfma32<DT>(sn, ka[s % KA], qop[s]);
#pragma unroll
            for (int i = s * 16 / SLOTS; i < (s + 1) * 16 / SLOTS; ++i) prob(i);
            KV_SB;
        }
        float mx = 0.f;
        static_assert(NCB >= 2, "three of out^T's instructions stand between the scores' last and their maximum");
        // (assembly: fmaxf quiets every matrix-core result first.  The compiler's hazard handling does not look into it: the
        // scores' last matrix-core instruction is two or more of out^T's behind, which issue one after the other)
        auto max_step = [&](int i) __attribute__((always_inline)) {
            if (i == 0) asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(mx) : "v"(sn[0]), "v"(sn[1]), "v"(sn[2]));
            else if (i < 7) asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(mx) : "v"(mx), "v"(sn[2 * i + 1]), "v"(sn[2 * i + 2]));
            else asm volatile("v_max_f32 %0, %1, %2" : "=v"(mx) : "v"(mx), "v"(sn[15]));
        };
        constexpr int NX = 2 * NCB;
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            if (x + AH < NX) read_v(x + AH);
            mfma32<DT>(oacc[x % NCB], va[x % VA], pb[x / NCB]);
            if (LM && x % NCB == 0) lacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones.h, pb[x / NCB].h, lacc, 0, 0, 0);
            if (KS + x < SLOTS) {
#pragma unroll
                for (int i = (KS + x) * 16 / SLOTS; i < (KS + x + 1) * 16 / SLOTS; ++i) prob(i);
            }
            KV_SB;
            if (x >= 2) {
#pragma unroll
                for (int i = (x - 2) * 8 / (NX - 2); i < (x - 1) * 8 / (NX - 2); ++i) max_step(i);
                KV_SB;
            }
        }
        need = __any(ef * mx > m_run + RAISE);
    };
    auto finish = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    if (nb > 0) {
        // block k's K lies in slot (k + 3) & 3 = (k - 1) & 3 of its ring, its V in slot k & 3
        request_k(0, 3);
        request_v(0, 0);
        request_k(1, 0);
        request_k(2, 1);
        request_v(1, 1);
    }
    if (flip) {
#pragma unroll
        for (int s = 0; s < KS; ++s) qop[s].v ^= u4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
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
        q_lo = any ? lo : 0x40000000;
        q_span = any ? (uint32_t)(hi - lo) : 0u;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // (in a form the compiler's bookkeeping sees)
    __syncthreads();
    if (nb > 0) {
        f16v sa, sb;
#pragma unroll
        for (int i = 0; i < 16; ++i) sa[i] = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            Op8 ka;
            ka.v = *reinterpret_cast<const u4 *>(kl + 3 * BLK + 2 * s * BN * 8);
            mfma32<DT>(sa, ka, qop[s]);
        }
        if (masked_block(0, 3)) apply_mask(0, 3, sa);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        int k = 0, s0 = 0;
        asm volatile("" : "+s"(k), "+s"(s0));  // (here and below: keeps the compiler from peeling an iteration, and its registers)  // s0: (k & 2), the ring half that blocks k + 1, k + 2 (K) and k, k + 1 (V) lie in
        bool need;
        auto requests = [&]() __attribute__((always_inline)) {
            const int o = s0 ^ 2;
            request_k(k + 3, o);
            request_k(k + 4, o + 1);
            request_v(k + 2, o);
            request_v(k + 3, o + 1);
        };
#pragma clang loop unroll(disable)
        for (;;) {
            // The fast loop holds neither masks nor rescaling: it is left when scores call for a higher reference maximum, in
            // the middle of an iteration (`mid`: block k + 1's are in sb) or at its end, or when a block needs its mask.
            do_raise(sa);
            bool mid = false;
            auto plain = [&]() __attribute__((always_inline)) -> bool {
                if (MM == 2 || k + 2 >= nb) return false;
                int m = masked_block(k + 1, s0) || masked_block(k + 2, s0 + 1);
                m = __builtin_amdgcn_readfirstlane(m);
                asm volatile("" : "+s"(m));
                return !m;
            };
            need = false;
#pragma clang loop unroll(disable)
            while (plain()) {
                requests();
                step(sa, sb, s0, need);
                if (need) {
                    mid = true;
                    break;
                }
                step(sb, sa, s0 + 1, need);
                finish();
                k += 2;
                s0 ^= 2;
                asm volatile("" : "+s"(k));
                if (need) break;
            }
            if (!mid && need) continue;
            if (!mid) {
                requests();
                step(sa, sb, s0, need);
                if (k + 1 >= nb) break;
                if (__builtin_amdgcn_readfirstlane(masked_block(k + 1, s0))) apply_mask(k + 1, s0, sb);
            }
            do_raise(sb);
            step(sb, sa, s0 + 1, need);
            if (k + 2 >= nb) break;
            if (__builtin_amdgcn_readfirstlane(masked_block(k + 2, s0 + 1))) apply_mask(k + 2, s0 + 1, sa);
            finish();
            k += 2;
            s0 ^= 2;
        }
    }
    else if (HV == 2) asm volatile("s_barrier" ::: "memory");
    if (HV == 2)
        for (int i = 0; i < idle; ++i) asm volatile("s_barrier" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (requests past the last block)

    // ---- the two halves' sums: each group ends with the whole of half of the columns ----
    constexpr int C0 = (NCB + 1) / 2;  // column blocks of the first group
    [[maybe_unused]] constexpr int WSZ = (C0 * 16 + 2) * 64;  // floats that a wavefront gives
    if constexpr (HV == 2) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the rings have been read
        float *const ex = reinterpret_cast<float *>(ring_s);
        float *mine = ex + wave8 * WSZ + lane, *other = ex + (wave8 ^ 4) * WSZ + lane;
        const float l_mine = LM ? (upper ? lacc[1] : lacc[0]) : l_run;
        mine[0] = m_run;
        mine[64] = l_mine;
        auto give = [&](auto C_, auto N_) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < decltype(N_)::value; ++c)
#pragma unroll
                for (int i = 0; i < 16; ++i) mine[(2 + c * 16 + i) * 64] = oacc[decltype(C_)::value + c][i];
        };
        auto take = [&](auto C_, auto N_, float mw, float ow) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < decltype(N_)::value; ++c)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    oacc[decltype(C_)::value + c][i] = oacc[decltype(C_)::value + c][i] * mw + other[(2 + c * 16 + i) * 64] * ow;
        };
        using Z = std::integral_constant<int, 0>;
        using C = std::integral_constant<int, C0>;
        using E = std::integral_constant<int, NCB - C0>;
        if (half) give(Z(), C());
        else give(C(), E());
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const float m_other = other[0], l_other = other[64], m = fmaxf(m_run, m_other);
        const float mw = m == -INFINITY ? 0.f : exp2_fast(m_run - m), ow = m == -INFINITY ? 0.f : exp2_fast(m_other - m);
        m_run = m;
        l_run = l_mine * mw + l_other * ow;
        if (half) take(C(), E(), mw, ow);
        else take(Z(), C(), mw, ow);
    }

    // ---- normalise and store: lane (n, hh) holds out[q = n][d = 32 c + 8 i + 4 hh + j] ----
    float l = l_run;
    if (LM && HV == 1) l = upper ? lacc[1] : lacc[0];
    if (!LM) l += __shfl_xor(l, 32);
    // Both go through LDS, a wavefront's own part of it, and leave it 16 bytes a lane along the rows.
    using Z = std::integral_constant<int, 0>;
    using C = std::integral_constant<int, C0>;
    using A = std::integral_constant<int, NCB>;
    using E = std::integral_constant<int, NCB - C0>;
    const int row0 = row - n;
    uint16_t *stage;
    if constexpr (HV == 1) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the rings have been read
        static_assert(4 * 32 * (D + 8) <= KSZ + VSZ && 4 * 32 * 36 * 2 <= KSZ + VSZ, "room for every wavefront's rows");
        stage = ring_s + wave * (32 * (D + 8 > 72 ? D + 8 : 72));
    } else {
        // (what the other group gave was for this wavefront alone, and it has read it)
        static_assert(32 * (32 * C0 + 8) <= 2 * WSZ && 32 * 36 <= WSZ, "room for a wavefront's rows");
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        stage = reinterpret_cast<uint16_t *>(reinterpret_cast<float *>(ring_s) + (wave8 ^ 4) * WSZ);
    }
    if (nsplit > 1) {
        // (from the registers 32 rows an instruction, of 32 bytes each: one sequence's 1024 new rows over 2000 keys in seven parts,
        // 8q/2kv x 128, 26.3 us the call for 24.2, and 25.8 on the tile before this one)
        float *part = a.workspace + (((size_t)bh * nsplit + item.split) * R + row0) * (D + 2), *fs = reinterpret_cast<float *>(stage);
        auto leave = [&](auto C_, auto N_) __attribute__((always_inline)) {  // column blocks C .. C + N - 1, one after the other
#pragma unroll
            for (int c = decltype(C_)::value; c < decltype(C_)::value + decltype(N_)::value; ++c) {
                const int W = 32 * c + 32 <= D ? 32 : 16, CPR = W / 4;
#pragma unroll
                for (int i = 0; i < W / 8; ++i)
                    *reinterpret_cast<f4 *>(fs + n * 36 + 8 * i + 4 * hh) = f4{oacc[c][4 * i], oacc[c][4 * i + 1], oacc[c][4 * i + 2], oacc[c][4 * i + 3]};
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (other lanes' columns: the order of the instructions is enough)
#pragma unroll
                for (int k = 0; k < CPR / 2; ++k) {
                    const int x = 64 * k + lane, rw = x / CPR, ch = x - rw * CPR;
                    if (row0 + rw < R) *reinterpret_cast<kv_part4 *>(part + rw * (D + 2) + 32 * c + 4 * ch) = *reinterpret_cast<const f4 *>(fs + rw * 36 + 4 * ch);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        };
        if constexpr (HV == 1) leave(Z(), A());
        else if (half) leave(C(), E());
        else leave(Z(), C());
        if (hh == 0 && half == 0 && q_ok) *reinterpret_cast<kv_f2 *>(part + n * (D + 2) + D) = kv_f2{m_run * 0.6931471805599453f, l};  // (the maximum back from the log2 domain)
        return;
    }
    // (8 bytes a lane from the registers are 32 rows an instruction, of 16 bytes each: where keys are few the launch was one of
    // such stores -- 16 prompts of 128, 32q/8kv x 128, bfloat16, the call 14.9 us for 12.3)
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    auto leave = [&](auto C_, auto N_) __attribute__((always_inline)) {
        constexpr int C = decltype(C_)::value, N = decltype(N_)::value, W = 32 * (C + N) < D ? 32 * N : D - 32 * C;
        constexpr int PITCH = W + 8, CPR = W / 8;  // 16-byte chunks of a row
#pragma unroll
        for (int c = 0; c < N; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (32 * c + 8 * i < W) {
                    const f16v &o = oacc[C + c];
                    const float o0 = o[4 * i] * inv, o1 = o[4 * i + 1] * inv, o2 = o[4 * i + 2] * inv, o3 = o[4 * i + 3] * inv;
                    *reinterpret_cast<kv_u2 *>(stage + n * PITCH + 32 * c + 8 * i + 4 * hh) =
                        DT == 1 ? kv_u2{pk_bf2(o0, o1), pk_bf2(o2, o3)} : kv_u2{pk_h2(o0, o1), pk_h2(o2, o3)};
                }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint16_t *op = reinterpret_cast<uint16_t *>(a.out) + ((size_t)bh * R + row0) * D + 32 * C;
#pragma unroll
        for (int k = 0; k < (32 * CPR + 63) / 64; ++k) {
            const int x = 64 * k + lane, rw = x / CPR, ch = x - rw * CPR;
            if (((32 * CPR) % 64 == 0 || x < 32 * CPR) && row0 + rw < R)
                *reinterpret_cast<kv_out8 *>(op + rw * D + 8 * ch) = *reinterpret_cast<const kv_u4 *>(stage + rw * PITCH + 8 * ch);
        }
    };
    if constexpr (HV == 1) leave(Z(), A());
    else if (half) leave(C(), E());
    else leave(Z(), C());
}

}  // namespace

// `halves`: workgroups of eight wavefronts, two groups of four that share the rows and halve the keys
hipError_t launch_attend_prefill_rows32(const AttendArgs &a, int nsplit, bool halves, hipStream_t s) {
    const Store &st = a.st;
    const int R = (a.Hq / a.Hkv) * a.L;
    dim3 grid((unsigned)((R + 127) / 128) * st.BH * nsplit);
    const bool ident = a.runs.n == 1 && a.runs.row0[0] == 0 && a.runs.phys0[0] == 0;
    const int mm = a.mask.mode == KVHIP_MASK_NONE ? 0 : (a.mask.mode == KVHIP_MASK_ARRAY ? 2 : 1);
#define P32_H(D, DT, ID, MM, HV) hipLaunchKernelGGL((prefill_rows32_kernel<D, DT, ID, MM, HV>), grid, dim3(256 * HV), 0, s, a, nsplit)
#define P32_M(D, DT, MM)                             \
    do {                                             \
        if (ident && halves) P32_H(D, DT, true, MM, 2);   \
        else if (ident) P32_H(D, DT, true, MM, 1);   \
        else if (halves) P32_H(D, DT, false, MM, 2); \
        else P32_H(D, DT, false, MM, 1);             \
    } while (0)
#define P32(D, DT)                      \
    do {                                \
        if (mm == 0) P32_M(D, DT, 0);   \
        else if (mm == 1) P32_M(D, DT, 1); \
        else P32_M(D, DT, 2);           \
    } while (0)
#define P32_DT(D)                               \
    do {                                        \
        if (st.dtype == KVHIP_F16) P32(D, 0);   \
        else P32(D, 1);                         \
    } while (0)
    if (st.Dk == 64) P32_DT(64);
    else if (st.Dk == 80) P32_DT(80);
    else if (st.Dk == 96) P32_DT(96);
    else P32_DT(128);
#undef P32_DT
#undef P32
#undef P32_M
#undef P32_H
    return hipGetLastError();
}

}  // namespace kvhip
