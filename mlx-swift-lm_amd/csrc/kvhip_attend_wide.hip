// Attention over 16-bit full-precision caches of head size 512 (Gemma 4's full-attention layers) on the matrix cores.
// The fused op (AttentionUtils.swift:86-93) computes in float32, excluded keys contribute nothing, one rounding at the
// output.
//
// A row of 512 is too wide for one wavefront's registers to hold queries, keys and outputs, so the four wavefronts of
// a workgroup divide the head dimension: wavefront w contracts elements 128 w .. 128 w + 127 of the scores and owns
// those columns of the output, and every cached element is loaded once per workgroup, from the page straight into the
// operand registers (the interleaved pages hold 8 elements of a token, or 8 tokens of a column, as one 16-byte chunk).
// Per tile of 32 tokens and 16 QT query rows:
//   S^T partials  K (32 tokens x 128) . Q^T on v_mfma_f32_16x16x32, into LDS, added up behind a barrier;
//   softmax       QT = 2: wavefronts 0 and 1 for sixteen query rows each, probabilities handed round through LDS;
//                 QT = 1: every wavefront for all sixteen rows (no second barrier);
//   out^T         V^T (128 columns x 32 tokens) . P^T, the probabilities as the sum of two 16-bit operands, high part
//                 and remainder: 22 bits of a float32 probability in float16 (scaled by 2^10, so that the remainder
//                 stays above the subnormals), 16 in bfloat16, where the output keeps 8.  Against float64 over 1 to
//                 512 rows and 333 to 8191 keys the outputs are off as with float32 probabilities (2.0 to 2.2 10^-4 and
//                 1.6 to 1.7 10^-3, equal to within 10^-5 of that).  An infinite value would meet a remainder of zero or of the
//                 other sign: where an output comes out NaN the workgroup goes over its keys again with the
//                 remainder's product over finite values only.
// Two rows of query tiles at most: the accumulators of four leave one wavefront per SIMD and are copied between the two
// register files every tile (512 rows x 2048 keys, 8 query and 2 kv heads, bfloat16: 69 us the call, against 57 us).
// Decode is bound by HBM where the batch fills the chip (B8, 4096 keys, one token: 26.5 us, 5.1 TB/s)
// and by launch, one pass of loads and the merge below that (one sequence of 2064 keys, the kernel 7.7 us with the rotation
// and the row's write, 10.4 before what its last workgroup and its first request waited for went, the merge 3.1; 63 us on the vector ALUs); a prompt chunk by the latency of the two barriers per tile
// (512 x 2048, 33 us on average over a prompt's chunks and 7.4 us for the merge; 263 us).
// K rows are loaded in the token order that leaves lane group g of the scores with tokens 8 g .. 8 g + 7, which is the
// order the probabilities are read in as an operand: they never cross lanes.
#include <algorithm>
#include <type_traits>

#include "kvhip_mask.hpp"
#include "kvhip_rope.hpp"

namespace kvhip {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int WD = 512;        // head size
constexpr int WW = 4;          // wavefronts
constexpr int WT = 32;         // tokens per tile
constexpr int NS = WD / WW / 32;  // contraction steps of a wavefront
constexpr int NCT = WD / WW / 16; // 16-column output tiles of a wavefront
constexpr float WLOG2E = 1.4426950408889634f;

template <int DT> __device__ __forceinline__ f4 mfma(const kv_u4 &a, const kv_u4 &b, f4 c) {
    if constexpr (DT == 0) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}
template <int DT> __device__ __forceinline__ uint32_t pack2(float x, float y) { return DT == 0 ? pk_h2(x, y) : pk_bf2(x, y); }
template <int DT> __device__ __forceinline__ float low_of(uint32_t w) {
    return DT == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)w) : __uint_as_float(w << 16);
}
template <int DT> __device__ __forceinline__ float high_of(uint32_t w) {
    return DT == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)) : __uint_as_float(w & 0xffff0000u);
}
// the elements of an operand that are finite, zeros for the others
template <int DT> __device__ __forceinline__ kv_u4 finite_only(kv_u4 v) {
    constexpr uint32_t E = DT == 0 ? 0x7c00u : 0x7f80u;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = ((v[i] & E) == E ? 0u : v[i] & 0xffffu) | ((v[i] & (E << 16)) == (E << 16) ? 0u : v[i] & 0xffff0000u);
    return v;
}

constexpr int SEEN = 4096;     // tiles of a part that a boolean mask is looked through for (131072 keys; beyond: taken as seen)

// grid (row blocks of 16 QT, BH, parts), four wavefronts.  Parts divide the key tiles the row block sees.
// ARR 1 / 2: boolean and additive array masks.  A row's elements are requested before the next tile's keys, whose arrival
// they would otherwise wait for; under a boolean mask the workgroup first looks which of its tiles any row sees and
// steps over the others, as the vector-ALU kernel does.  (All four wavefronts go by one table in LDS: they meet in the
// loop's barriers.)  One token, B8, 16q/8kv, 8192 keys: all seen under a boolean mask 212 us, a window of 512 47, an
// additive mask 193; 275, 276 and 262 with the elements fetched one by one behind the keys and every tile read, 198, 66
// and 193 on the vector-ALU kernel.
// A single-token step without a mask: the workgroup whose part holds the new row's tile writes the row, each wavefront
// its quarter.  If that tile is its first, as in the steps of a single sequence, the row goes into the tile's registers too.  ROT
// turns the query rows and the new key row in LDS first, as the decode kernels do.  A launch that appends takes 5.2 us.
template <int DT, int QT, int ARR, bool ROT>
__global__ void __launch_bounds__(256, 2)
attend_wide_kernel(typename DecodeArgs<ROT ? 3 : 0>::type a, int r, int tiles_total, int nparts) {
    constexpr int NB = QT == 1 ? 2 : 1;           // score buffers (QT = 1 has one barrier per tile)
    __shared__ f4 part_s[NB][WW][QT][2][64];      // partial scores of the wavefronts
    __shared__ kv_u4 prob_s[QT == 1 ? 1 : QT][2][64];
    __shared__ float stat_s[QT][16], sum_s[QT][16], max_s[QT][16];
    __shared__ int nan_s[WW];
    __shared__ uint8_t seen_s[ARR == 1 ? SEEN : 1];
    constexpr bool STEP = QT == 1 && ARR == 0;  // (up to 16 query rows: one row block)
    __shared__ __align__(16) uint16_t rot_s[ROT ? 17 * WD : 1];
    const Store &st = a.st;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, g = lane >> 4;
    const RowBlock rb(a);
    const int bh = rb.bh, part = rb.part, b = rb.b, h = rb.h;
    const int R = r * a.L;
    const int row0 = rb.block * 16 * QT, row1 = min(row0 + 16 * QT, R) - 1;

    // ---- the keys this row block sees ---------------------------------------------------------------
    const bool one_head = rb.head(row0) == rb.head(row1);
    const KeyRange keys = visible_keys(a.mask, b, a.L, a.T, one_head ? rb.pos(row0) : 0, one_head ? rb.pos(row1) : a.L - 1);
    const bool ident = a.runs.n == 1 && a.runs.row0[0] == 0 && a.runs.phys0[0] == 0;
    int t_lo = 0, t_hi = tiles_total;
    if (ident) {
        t_lo = min(keys.lo / WT, tiles_total);
        t_hi = keys.hi < keys.lo ? t_lo : min(tiles_total, keys.hi / WT + 1);
    }
    const int per = (max(t_hi - t_lo, 1) + nparts - 1) / nparts;
    const int tb = min(t_lo + part * per, t_hi), te = min(tb + per, t_hi);

    // ---- a step's rows ----------------------------------------------------------------------------------------
    [[maybe_unused]] RopeStep<DT, WD, 256, 16> step;
    if constexpr (ROT)
        step.fetch(a.turn, reinterpret_cast<const uint16_t *>(a.q) + (size_t)(b * a.Hq + h * r) * WD,
                   static_cast<const uint16_t *>(a.new_k) + (size_t)bh * WD, R);
    // (lane (col, g): the row's elements that its key operands of the row's token hold, and its values of columns 16 c + col)
    bool owner = false;  // workgroup-uniform
    kv_u4 own_k[NS];
    uint16_t own_v[NCT];
    if constexpr (STEP) {
        owner = a.new_k != nullptr && a.new_slot / WT >= tb && a.new_slot / WT < te;
        if (owner) {
#pragma unroll
            for (int s = 0; s < (ROT ? 0 : NS); ++s) own_k[s] = ld_global<kv_u4>(as_global(a.new_k) + ((size_t)bh * WD + wave * (WD / WW) + 8 * g + 32 * s) * 2);
#pragma unroll
            for (int c = 0; c < NCT; ++c) own_v[c] = ld_global<uint16_t>(as_global(a.new_v) + ((size_t)bh * WD + wave * (WD / WW) + 16 * c + col) * 2);
        }
    }
    auto write_row = [&](const PageEntry &page) __attribute__((always_inline)) {
        // (global stores: behind one to a plain pointer every load in flight is waited for)
        const int slot = a.new_slot, c0 = wave * (WD / WW);
        KV_GLOBAL char *kc = (KV_GLOBAL char *)as_global(page.k + (size_t)bh * st.k_cell), *vc = (KV_GLOBAL char *)as_global(page.v + (size_t)bh * st.v_cell);
        if (col == 0) {
#pragma unroll
            for (int s = 0; s < NS; ++s) *reinterpret_cast<KV_GLOBAL kv_u4 *>(kc + kfp_at<2>(2 * WD, slot, c0 + 8 * g + 32 * s)) = own_k[s];
        }
        if (g == 0) {
#pragma unroll
            for (int c = 0; c < NCT; ++c) *reinterpret_cast<KV_GLOBAL uint16_t *>(vc + vfp_at<2>(WD, slot, c0 + 16 * c + col)) = own_v[c];
        }
    };
    auto row_written = []() __attribute__((always_inline)) {  // (a wavefront reads the quarter that it wrote)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };

    // ---- query operands: lane (col, g) holds elements 8 g .. 8 g + 7 of step s of row 16 qt + col ----
    kv_u4 qop[QT][NS];
#pragma unroll
    for (int qt = 0; qt < (ROT ? 0 : QT); ++qt) {
        const int rr = min(row0 + 16 * qt + col, R - 1);  // rows beyond the last: the last again, which nobody keeps
        gptr qp = as_global(a.q) + (((size_t)(b * a.Hq + h * r + rb.head(rr)) * a.L + rb.pos(rr)) * WD + wave * (WD / WW) + 8 * g) * 2;
#pragma unroll
        for (int s = 0; s < NS; ++s) qop[qt][s] = ld_global<kv_u4>(qp + s * 64);
    }

    kv_u4 kreg[NS][2], vreg[NCT];
    const uint32_t k_lane = ((uint32_t)(16 * wave + g) * TILE + 8 * (col >> 2) + (col & 3)) * 16;
    const uint32_t v_lane = ((uint32_t)g * WD + wave * (WD / WW) + col) * 16;
    PageCursor kpage(st, tb < te ? tb * WT : 0), vpage = kpage;
    auto load_k = [&](int t) __attribute__((always_inline)) {
        const int slot0 = t * WT;
        gptr p = as_global(kpage.at(st, slot0).k) + (size_t)bh * st.k_cell + (size_t)((slot0 & (PAGE - 1)) >> 6) * ((size_t)TILE * st.k_row) +
                 (slot0 & 32) * 16 + k_lane;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int x = 0; x < 2; ++x) kreg[s][x] = ld_global<kv_u4>(p + s * (4 * TILE * 16) + x * 64);
    };
    auto load_v = [&](int t) __attribute__((always_inline)) {
        const int slot0 = t * WT;
        gptr p = as_global(vpage.at(st, slot0).v) + (size_t)bh * st.v_cell + (size_t)((slot0 & (PAGE - 1)) >> 6) * ((size_t)TILE * WD * 2) +
                 (size_t)((slot0 & 32) >> 3) * (WD * 16) + v_lane;
#pragma unroll
        for (int c = 0; c < NCT; ++c) vreg[c] = ld_global<kv_u4>(p + c * 256);
    };

    f4 acc[QT][NCT];
    const int own = QT == 1 ? 0 : wave & 1;  // the query rows whose softmax this wavefront works out
    const int my = row0 + 16 * own + col;
    const int my_hq = h * r + rb.head(min(my, R - 1)), my_l = rb.pos(min(my, R - 1));
    float m_run, l_run;
    constexpr float P_UP = DT == 0 ? 10.f : 0.f;  // (float16 probabilities are carried times 2^10)

    // (1) the first tile from t on that a row sees
    if constexpr (ARR == 1) {
        constexpr int U = 4;  // tiles a wavefront asks for together
        const int n = min(te - tb, SEEN);
        for (int i0 = wave; i0 < n; i0 += U * WW) {
            uint32_t w[U][QT][2];
            bool seen[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int slot0 = (tb + min(i0 + u * WW, n - 1)) * WT, row = run_row(a.runs, slot0, WT);
                seen[u] = false;
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    const int rr = min(row0 + 16 * qt + col, R - 1), hq = h * r + rr / a.L, l = rr % a.L;
                    w[u][qt][0] = w[u][qt][1] = 0u;
                    if (row >= 0) {
                        mask_bool_words<2>(a.mask, b, hq, l, row + 8 * g, w[u][qt]);
                    } else {
                        for (int j = 0; j < 8; ++j) {
                            const int slot = slot0 + 8 * g + j, key = slot < a.slots ? slot_to_row(a.runs, slot) : -1;
                            float add;
                            seen[u] = seen[u] || (key >= 0 && key < a.T && mask_keep(a.mask, b, hq, l, key, a.L, a.T, add));
                        }
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) seen[u] = seen[u] || (w[u][qt][0] | w[u][qt][1]) != 0u;
                const bool any = __any(seen[u]);
                if (lane == 0 && i0 + u * WW < n) seen_s[i0 + u * WW] = any;
            }
        }
        __syncthreads();
    }
    auto seen_from = [&](int t) __attribute__((always_inline)) -> int {
        if constexpr (ARR == 1) {
            while (t < te && t - tb < SEEN) {
                const int i = t - tb + lane;
                const unsigned long long m = __ballot(t + lane < te && (i >= SEEN || seen_s[min(i, SEEN - 1)] != 0));
                if (m != 0ull) return t + __ffsll(m) - 1;
                t += 64;
            }
            return min(t, te);
        }
        return t;
    };
    uint32_t raw[ARR == 1 ? 2 : 8];  // (ARR) the mask elements of row `my` for tokens 8 g .. 8 g + 7 of a tile
    auto mask_fetch = [&](int t) __attribute__((always_inline)) {
        const int row = run_row(a.runs, t * WT, WT);
        if (row < 0 || (QT > 1 && wave >= QT)) return;
        if constexpr (ARR == 1) mask_bool_words<2>(a.mask, b, my_hq, my_l, row + 8 * g, raw);
        if constexpr (ARR == 2) mask_add_words<8>(a.mask, b, my_hq, my_l, row + 8 * g, raw);
    };

    // the probabilities of row `my` for tokens 8 g .. 8 g + 7 of tile t, high parts and remainders, and the factor its
    // sums so far take
    auto softmax = [&](auto careful, int t, int buf, kv_u4 &ph, kv_u4 &pl, float &alpha) __attribute__((always_inline)) {
        f4 sum[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            sum[x] = part_s[buf][0][own][x][lane];
#pragma unroll
            for (int w = 1; w < WW; ++w) sum[x] += part_s[buf][w][own][x][lane];
        }
        float sc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) sc[j] = sum[j >> 2][j & 3] * a.scale;
        const int slot0 = t * WT;
        if (ARR != 0 && run_row(a.runs, slot0, WT) >= 0) {  // workgroup-uniform
            if constexpr (ARR == 1) {
#pragma unroll
                for (int j = 0; j < 8; ++j) sc[j] = ((raw[j >> 2] >> (8 * (j & 3))) & 0xffu) != 0u ? sc[j] : -INFINITY;
            } else if constexpr (ARR == 2) {
                float add[8];
                mask_add_floats<8>(a.mask, raw, add);
#pragma unroll
                for (int j = 0; j < 8; ++j) sc[j] += add[j];
            }
        } else if (QT == 1 && ARR == 0 && rb.one && ident) {  // one token: every row sees keys.lo to keys.hi
            // (evaluated key by key as below, the tile at the edge, a step's last, took 2.5 us longer than the others)
            if (slot0 < keys.lo || slot0 + WT - 1 > keys.hi) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int row = slot0 + 8 * g + j;
                    sc[j] = row >= keys.lo && row <= keys.hi ? sc[j] : -INFINITY;
                }
            }
        } else if (!ident || slot0 < keys.full_lo || slot0 + WT - 1 > keys.full_hi) {  // workgroup-uniform
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int slot = slot0 + 8 * g + j;
                const int row = ident ? slot : slot < a.slots ? slot_to_row(a.runs, slot) : -1;
                float add = 0.f;
                const bool keep = row >= 0 && row < a.T && mask_keep(a.mask, b, my_hq, my_l, row, a.L, a.T, add);
                sc[j] = keep ? sc[j] + add : -INFINITY;
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            sc[j] = fmaxf(sc[j], -INFINITY);  // (a score that is NaN weighs nothing)
            mx = fmaxf(mx, sc[j]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // The reference of the exponentials is raised only when a score exceeds it by more than 2^5, so that the
        // accumulators are rarely touched after the first tiles (probabilities stay below 2^5, 2^15 in float16).
        const float m_new = (mx - m_run) * WLOG2E > 5.f || m_run == -INFINITY ? fmaxf(m_run, mx) : m_run;
        const float m_use = m_new > -INFINITY ? m_new : 0.f;
        alpha = m_new > m_run ? __builtin_amdgcn_exp2f((m_run - m_new) * WLOG2E) : 1.f;
        float p[8], ps = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j] - m_use, WLOG2E, P_UP));
            ps += p[j];
        }
        l_run = l_run * alpha + ps;
        m_run = m_new;
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            hi[j] = pack2<DT>(p[2 * j], p[2 * j + 1]);
            if constexpr (DT == 0 && decltype(careful)::value) {  // no weight rounds to nothing (the remainder takes it off again)
                if (p[2 * j] > 0.f && (hi[j] & 0xffffu) == 0u) hi[j] |= 1u;
                if (p[2 * j + 1] > 0.f && (hi[j] >> 16) == 0u) hi[j] |= 0x10000u;
            }
            lo[j] = pack2<DT>(p[2 * j] - low_of<DT>(hi[j]), p[2 * j + 1] - high_of<DT>(hi[j]));
        }
        ph = kv_u4{hi[0], hi[1], hi[2], hi[3]};
        pl = kv_u4{lo[0], lo[1], lo[2], lo[3]};
    };

    // Behind a part's last tile, often a step's only one, the tile is not requested again; long loops keep their requests in front
    // of no branch (512 rows over 3000 keys, B4, 8q/2kv: 188 us with one, 183 without).
    constexpr bool BRANCH = QT == 1;
    // All the keys; true if an output came out NaN (`careful`: infinite values are about).
    auto walk = [&](auto careful) __attribute__((always_inline)) {
        m_run = -INFINITY;
        l_run = 0.f;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int c = 0; c < NCT; ++c) acc[qt][c] = f4{0.f, 0.f, 0.f, 0.f};
        int t = seen_from(tb), buf = 0;
        if (t < te && (decltype(careful)::value || !STEP)) {  // workgroup-uniform
            load_k(t);
            load_v(t);
        }
        while (t < te) {
            const int next = seen_from(t + 1);
            if constexpr (ARR != 0) mask_fetch(t);
            f4 sacc[QT][2];
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) sacc[qt][0] = sacc[qt][1] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                    for (int x = 0; x < 2; ++x) sacc[qt][x] = mfma<DT>(kreg[s][x], qop[qt][s], sacc[qt][x]);
            if (!BRANCH || next < te) load_k(next < te ? next : t);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                for (int x = 0; x < 2; ++x) part_s[buf][wave][qt][x][lane] = sacc[qt][x];
            __syncthreads();
            kv_u4 ph, pl;
            float alpha = 1.f;
            if (QT == 1 || wave < QT) softmax(careful, t, buf, ph, pl, alpha);  // wave-uniform
            if constexpr (QT > 1) {
                if (wave < QT) {
                    prob_s[own][0][lane] = ph;
                    prob_s[own][1][lane] = pl;
                    if (g == 0) stat_s[own][col] = alpha;
                }
                __syncthreads();
            }
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                const float al = QT == 1 ? alpha : stat_s[qt][col];
                if (__any(al != 1.f)) {  // (a raised maximum: rare after the first tiles)
#pragma unroll
                    for (int c = 0; c < NCT; ++c) acc[qt][c] *= al;
                }
                if constexpr (QT > 1) {
                    ph = prob_s[qt][0][lane];
                    pl = prob_s[qt][1][lane];
                }
#pragma unroll
                for (int c = 0; c < NCT; ++c) acc[qt][c] = mfma<DT>(vreg[c], ph, acc[qt][c]);
#pragma unroll
                for (int c = 0; c < NCT; ++c) acc[qt][c] = mfma<DT>(decltype(careful)::value ? finite_only<DT>(vreg[c]) : vreg[c], pl, acc[qt][c]);
            }
            if (!BRANCH || next < te) load_v(next < te ? next : t);
            t = next;
            buf ^= NB - 1;
        }

        // ---- the rows' maxima and sums to every wavefront ----------------------------------------------
        l_run += __shfl_xor(l_run, 16);
        l_run += __shfl_xor(l_run, 32);
        f4 probe = acc[0][0];  // (a sum: NaN where one of them is; infinities of both signs only cost the second walk)
#pragma unroll
        for (int i = 1; i < QT * NCT; ++i) probe += acc[i / NCT][i % NCT];
        const float probed = (probe.x + probe.y) + (probe.z + probe.w);
        const bool nan = __any(probed != probed);
        if (lane == 0) nan_s[wave] = nan;
        if (g == 0 && wave < QT) {
            max_s[own][col] = m_run;
            sum_s[own][col] = l_run;
        }
        __syncthreads();
        return (nan_s[0] | nan_s[1] | nan_s[2] | nan_s[3]) != 0;  // workgroup-uniform
    };
    if constexpr (STEP) {  // (ahead of the first walk: the row is written, and the rows turned, meanwhile)
        if (tb < te) {
            load_k(tb);
            load_v(tb);
        }
        if constexpr (ROT) {
            step.turn(a.turn, bh, R, rot_s);
            __syncthreads();
            const uint16_t *qr = rot_s + min(row0 + col, R - 1) * WD + wave * (WD / WW) + 8 * g;
#pragma unroll
            for (int s = 0; s < NS; ++s) qop[0][s] = *reinterpret_cast<const kv_u4 *>(qr + 32 * s);
        }
        if (owner) {
            if constexpr (ROT) {
#pragma unroll
                for (int s = 0; s < NS; ++s) own_k[s] = *reinterpret_cast<const kv_u4 *>(rot_s + R * WD + wave * (WD / WW) + 8 * g + 32 * s);
            }
            PageCursor page = kpage;
            write_row(page.at(st, a.new_slot));
            // (only a tile that is still to be read has to wait for the row: behind a fence and with the page looked up again
            // a step's last workgroup ended 3 us behind the others)
            if (a.new_slot / WT != tb) {
                row_written();
            } else {
                const int tn = a.new_slot & (WT - 1);  // token 8 (c / 4) + 4 x + c % 4 is operand row c of block x
                const bool mine = col == 4 * (tn >> 3) + (tn & 3);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int x = 0; x < 2; ++x) kreg[s][x] = mine && ((tn >> 2) & 1) == x ? own_k[s] : kreg[s][x];
#pragma unroll
                for (int c = 0; c < NCT; ++c)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {  // value tn % 8 of the lane's eight, if they are token tn's
                        const uint32_t old = vreg[c][w];
                        const uint32_t both = (tn & 1) ? (old & 0xffffu) | ((uint32_t)own_v[c] << 16) : (old & 0xffff0000u) | own_v[c];
                        vreg[c][w] = g == tn >> 3 && w == ((tn & 7) >> 1) ? both : old;
                    }
            }
        }
    }
    const bool again = walk(std::false_type());
    if (__builtin_expect(again, 0)) {
        if (owner) row_written();
        __syncthreads();
        walk(std::true_type());
    }

#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int rr = row0 + 16 * qt + col;
        if (rr >= R) continue;
        const float l = sum_s[qt][col];
        if (nparts == 1) {
            const float inv = l > 0.f ? 1.f / l : 0.f;
            uint16_t *dst = reinterpret_cast<uint16_t *>(a.out) + ((size_t)(b * a.Hq + h * r + rb.head(rr)) * a.L + rb.pos(rr)) * WD + wave * (WD / WW) + 4 * g;
#pragma unroll
            for (int c = 0; c < NCT; ++c) {
                const f4 v = acc[qt][c] * inv;
                *reinterpret_cast<kv_out4 *>(dst + 16 * c) = kv_out4{pack2<DT>(v.x, v.y), pack2<DT>(v.z, v.w)};
            }
        } else {
            float *dst = a.workspace + ((size_t)(bh * nparts + part) * R + rr) * (WD + 2);
#pragma unroll
            for (int c = 0; c < NCT; ++c) {
                float *d = dst + wave * (WD / WW) + 16 * c + 4 * g;  // (rows of 514 floats: 8-byte aligned)
                *reinterpret_cast<kv_f2 *>(d) = kv_f2{acc[qt][c].x, acc[qt][c].y};
                *reinterpret_cast<kv_f2 *>(d + 2) = kv_f2{acc[qt][c].z, acc[qt][c].w};
            }
            if (wave == 0 && g == 0) {
                dst[WD] = max_s[qt][col];
                dst[WD + 1] = l;
            }
        }
    }
}

struct PlanWide {
    int qt, row_blocks, tiles, nparts;
};

PlanWide plan_wide(const AttendArgs &a) {
    PlanWide p;
    const int R = (a.Hq / a.Hkv) * a.L;
    p.qt = R <= 16 ? 1 : 2;
    p.row_blocks = (R + 16 * p.qt - 1) / (16 * p.qt);
    p.tiles = (a.slots + WT - 1) / WT;
    // One token: a workgroup per CU (two: B8 over 4096 keys 29.4 us against 26.8), parts of a tile and up (two: 11.2 us against
    // 10.1 for a sequence of 2048 keys, the merge, which has every part's loads in flight at once, 3.5 us for either), but
    // up to three tiles one part, without a merge (a step of 60 keys 12.6 us against 14.4, of 90 13.7 against 14.5).
    // Chunks: two per CU (one: 76 us against 57 for 512 x 2048; three, which need a second round: 72 us).
    static const int target = measure_knob("KVHIP_WIDE_TARGET", 256), target2 = measure_knob("KVHIP_WIDE_TARGET2", 512), least = measure_knob("KVHIP_WIDE_LEAST", 1);  // (timing builds only)
    const long wgs = (long)p.row_blocks * a.st.BH;
    int n = p.qt == 1 && p.tiles <= 3 ? 1 : (int)std::max(1L, std::min<long>((p.qt == 1 ? target : target2) / std::max(1L, wgs), p.tiles / (p.qt == 1 ? least : 4)));
    n = std::min(n, p.qt == 1 ? 128 : 64);
    const size_t per_part = (size_t)a.st.BH * R * (a.st.Dv + 2) * sizeof(float);
    while (n > 1 && a.workspace_cap && per_part * n > a.workspace_cap) --n;
    p.nparts = n;
    return p;
}

}  // namespace

bool attend_wide_supported(const AttendArgs &a) {
    const Store &s = a.st;
    return s.bits == 0 && s.es == 2 && s.Dk == WD && s.Dv == WD && s.BH <= 65535;
}

size_t attend_wide_workspace(const AttendArgs &a) {
    const PlanWide p = plan_wide(a);
    return p.nparts == 1 ? 0 : (size_t)a.st.BH * p.nparts * (a.Hq / a.Hkv) * a.L * (a.st.Dv + 2) * sizeof(float);
}

hipError_t launch_attend_wide(const AttendArgs &a, hipStream_t s) {
    const PlanWide p = plan_wide(a);
    const dim3 grid(p.row_blocks, a.st.BH, p.nparts), block(256);
    profile_mark(s, true);
    const int arr = a.mask.mode != KVHIP_MASK_ARRAY ? 0 : a.mask.dtype == KVHIP_BOOL ? 1 : 2;
#define WIDE_A(DT, QT, ARR) hipLaunchKernelGGL((attend_wide_kernel<DT, QT, ARR, false>), grid, block, 0, s, a, a.Hq / a.Hkv, p.tiles, p.nparts)
#define WIDE(DT, QT)                       \
    do {                                   \
        if (QT == 1 && a.new_k && a.rope)  \
            hipLaunchKernelGGL((attend_wide_kernel<DT, 1, 0, true>), grid, block, 0, s, AttendStepArgs(a), a.Hq / a.Hkv, p.tiles, p.nparts); \
        else if (arr == 0) WIDE_A(DT, QT, 0); \
        else if (arr == 1) WIDE_A(DT, QT, 1); \
        else WIDE_A(DT, QT, 2);            \
    } while (0)
    if (a.st.dtype == KVHIP_F16) {
        if (p.qt == 1) WIDE(0, 1);
        else WIDE(0, 2);
    } else {
        if (p.qt == 1) WIDE(1, 1);
        else WIDE(1, 2);
    }
#undef WIDE
#undef WIDE_A
    profile_mark(s, false);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.nparts == 1) return e;
    return launch_merge_valu(a, p.nparts, s);
}

}  // namespace kvhip
