// Attention over float32 caches on the float32 matrix instruction (v_mfma_f32_16x16x4_f32: products and sums in
// float32, twice the rate of the vector ALUs).  The fused op (AttentionUtils.swift:86-93): excluded keys contribute
// nothing, no rounding but float32's.
//
// A workgroup takes 16 QT query rows of one kv head and one range of keys; its four wavefronts walk alternate tiles of
// 16 TB tokens with their own maxima, sums and accumulators and meet once, through LDS, at the end.  Nothing crosses
// lanes in the loop but the row maxima, because the interleaved pages hold what each operand wants:
//   S^T = K Q^T    lane (i, g) loads 16 bytes, elements 16 s + 4 g .. + 3 of token i: its operand of four instructions
//                  (instruction j contracts elements 16 s + 4 g + j, g = 0..3), the queries likewise from their rows;
//   out^T = V^T P^T  lane (i, g) loads tokens 4 g .. 4 g + 3 of column i, and the scores leave the first product with
//                  tokens 4 g .. 4 g + 3 of query i in lane (i, g): the probabilities are the operand as they are.
// Measured against the vector-ALU kernel, whole calls: 512 x 4096, B4, 32q/8kv 1626 -> 654 us (D 64), 2644 -> 1215
// (D 128: 106 TFLOP/s of the 157 that the instruction has), 6755 -> 2480 (D 256); one token of one sequence, 16q/4kv, 1500
// keys 17.3 -> 9.9 us (D 64: one pass of loads, 6.4, and the merge, 3.5); 8192 keys of B8, 8 kv heads, HBM: 102 -> 101 us (D 128).
#include <algorithm>

#include "kvhip_mask.hpp"
#include "kvhip_rope.hpp"

namespace kvhip {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int MW = 4;  // wavefronts

__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// token blocks of 16 per tile: as many as the registers of two wavefronts per SIMD hold
constexpr int token_blocks(int dk, int qt) { return dk <= 64 ? 4 / qt : dk <= 128 ? 2 / qt : 1; }
constexpr int query_tiles(int dk) { return dk <= 128 ? 2 : 1; }

// grid (row blocks of 16 QT, BH, parts).  Parts divide the key tiles the row block sees.
// ARR 1 / 2: boolean and additive array masks.  Their elements are requested before the next tile's keys, whose arrival
// they would otherwise wait for, and a wavefront steps over tiles that none of its rows sees under a boolean one, as
// those of the vector-ALU kernel do.
// One token, B8, 32q/8kv, D 128, 8192 keys: all seen under a boolean mask 107 us, a window of 512 31, an additive mask
// 104; 119, 120 and 112 with the elements fetched one by one behind the keys and every tile read, 105, 43 and 100 on
// the vector-ALU kernel; 256 rows of B4 over 4096 keys, the boolean window: 236, 893, 476.
// A single-token step without a mask: the wavefront that reads the new row's tile writes the row after it has requested
// its first tile -- and if that is the row's tile, puts the row into its registers too --, and ROT turns the query rows and
// the new key row in LDS first, as the decode kernels do.  A launch that appends takes 4.2 us.
// TB: token blocks of 16 per tile.  ONE: it may be a single token (head sizes above 128, where prompt chunks take one query tile
// too, have an instance of its own for it): what only a token needs is not in the loop of prompt chunks, where it cost them 1 to
// 2 % (16q/4kv x 64, 512 rows over 2048 keys 52.5 us for 51.5, over 6000 133.9 for 132.2; 192 / 128 103.8 for 102.2).
template <int DK, int DV, int QT, int TB, int ARR, bool ROT, bool ONE>
__global__ void __launch_bounds__(256, 2)
attend_f32_kernel(typename DecodeArgs<ROT ? 3 : 0>::type a, int r, int tiles_total, int nparts) {
    constexpr int WT = 16 * TB;
    constexpr int NS = DK / 16, NCT = DV / 16;
    extern __shared__ __align__(16) float smem[];
    f4 *acc_s = reinterpret_cast<f4 *>(smem);         // [MW][QT][NCT][64]
    constexpr bool QL = DK > 128;                     // query operands in LDS: no registers are left for them
    f4 *q_s = reinterpret_cast<f4 *>(smem);           // [QT][NS][64], where the accumulators go after the loop: beside them
                                                      // only one workgroup of head size 256 would fit a CU (that call: 2607)
    __shared__ float max_s[MW][QT][16], sum_s[MW][QT][16];
    const Store &st = a.st;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, g = lane >> 4;
    const RowBlock rb(a);
    const int bh = rb.bh, part = rb.part, b = rb.b, h = rb.h;
    const int R = r * a.L;
    const int row0 = rb.block * 16 * QT, row1 = min(row0 + 16 * QT, R) - 1;

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
    constexpr bool STEP = QT == 1 && ARR == 0 && ONE;  // (up to 16 query rows: one row block)
    // (behind a wavefront's last tile, often a step's only one, the tile is not requested again; long loops keep their requests
    // in front of no branch)
    constexpr bool BRANCH = STEP && !QL;
    float *rot_s = smem + (QL ? NS * 256 : 0);  // [R + 1][DK] behind the query operands, under what the accumulators take at the end
    static_assert((QL ? NS * 256 : 0) + 17 * DK <= MW * NCT * 256, "room for sixteen query rows and the key row");
    [[maybe_unused]] RopeStep<2, DK, 256, 16> step;
    if constexpr (ROT)
        step.fetch(a.turn, static_cast<const float *>(a.q) + (size_t)(b * a.Hq + h * r) * DK, static_cast<const float *>(a.new_k) + (size_t)bh * DK, R);
    // (lane (col, g): the row's elements that its key operands of the row's token hold, and its values of columns 16 c + col)
    bool own = false;  // wave-uniform
    f4 own_k[NS];
    float own_v[NCT];
    if constexpr (STEP) {
        const int tn = a.new_slot / WT;
        own = a.new_k != nullptr && tn >= tb && tn < te && (tn - tb) % MW == wave;
        if (own) {
#pragma unroll
            for (int s = 0; s < (ROT ? 0 : NS); ++s) own_k[s] = ld_global<f4>(as_global(a.new_k) + ((size_t)bh * DK + 16 * s + 4 * g) * 4);
#pragma unroll
            for (int c = 0; c < NCT; ++c) own_v[c] = ld_global<float>(as_global(a.new_v) + ((size_t)bh * DV + 16 * c + col) * 4);
        }
    }
    auto write_row = [&](const PageEntry &page) __attribute__((always_inline)) {
        if constexpr (ROT) {
#pragma unroll
            for (int s = 0; s < NS; ++s) own_k[s] = *reinterpret_cast<const f4 *>(rot_s + R * DK + 16 * s + 4 * g);
        }
        // (global stores: see attend_wide_kernel)
        const int slot = a.new_slot;
        KV_GLOBAL char *kc = (KV_GLOBAL char *)as_global(page.k + (size_t)bh * st.k_cell), *vc = (KV_GLOBAL char *)as_global(page.v + (size_t)bh * st.v_cell);
        if (col == 0) {
#pragma unroll
            for (int s = 0; s < NS; ++s) *reinterpret_cast<KV_GLOBAL f4 *>(kc + kfp_at<4>(4 * DK, slot, 16 * s + 4 * g)) = own_k[s];
        }
        if (g == 0) {
#pragma unroll
            for (int c = 0; c < NCT; ++c) *reinterpret_cast<KV_GLOBAL float *>(vc + vfp_at<4>(DV, slot, 16 * c + col)) = own_v[c];
        }
    };

    // rows beyond the last: the last again, which nobody keeps
    f4 qop[QT][QL ? 1 : NS];
    int my_hq[QT], my_l[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int rr = min(row0 + 16 * qt + col, R - 1);
        my_hq[qt] = h * r + rb.head(rr);
        my_l[qt] = rb.pos(rr);
        gptr qp = as_global(a.q) + (((size_t)(b * a.Hq + my_hq[qt]) * a.L + my_l[qt]) * DK + 4 * g) * 4;
#pragma unroll
        for (int s = 0; s < (QL || ROT ? 0 : NS); ++s) qop[qt][s] = ld_global<f4>(qp + s * 64);
        if constexpr (QL && !ROT) {
            for (int s = wave; s < NS; s += MW) q_s[(qt * NS + s) * 64 + lane] = ld_global<f4>(qp + s * 64);
        }
    }
    if constexpr (QL && !ROT) __syncthreads();

    f4 kreg[TB][NS], vreg[TB][NCT];
    const uint32_t k_lane = ((uint32_t)g * TILE + col) * 16, v_lane = ((uint32_t)g * DV + col) * 16;
    const int first = tb + wave;
    PageCursor kpage(st, first < te ? first * WT : 0), vpage = kpage;
    auto load_k = [&](int t) __attribute__((always_inline)) {
        const int slot0 = t * WT;
        gptr p = as_global(kpage.at(st, slot0).k) + (size_t)bh * st.k_cell + (size_t)((slot0 & (PAGE - 1)) >> 6) * (TILE * DK * 4) +
                 (slot0 & 63) * 16 + k_lane;
#pragma unroll
        for (int x = 0; x < TB; ++x)
#pragma unroll
            for (int s = 0; s < NS; ++s) kreg[x][s] = ld_global<f4>(p + s * (4 * TILE * 16) + x * 256);
    };
    auto load_v = [&](int t) __attribute__((always_inline)) {
        const int slot0 = t * WT;
        gptr p = as_global(vpage.at(st, slot0).v) + (size_t)bh * st.v_cell + (size_t)((slot0 & (PAGE - 1)) >> 2) * (DV * 16) + v_lane;
#pragma unroll
        for (int x = 0; x < TB; ++x)
#pragma unroll
            for (int c = 0; c < NCT; ++c) vreg[x][c] = ld_global<f4>(p + x * (4 * DV * 16) + c * 256);
    };

    f4 acc[QT][NCT];
    float m_run[QT], l_run[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        m_run[qt] = -INFINITY;
        l_run[qt] = 0.f;
#pragma unroll
        for (int c = 0; c < NCT; ++c) acc[qt][c] = f4{0.f, 0.f, 0.f, 0.f};
    }
    // (ARR) the raw mask elements of a tile, and (1) which of the lane's keys its rows see, bit (qt TB + x) 4 + j
    constexpr bool bools = ARR == 1;
    uint32_t raw[QT][TB][bools ? 1 : 4];
    auto mask_fetch = [&](int t) __attribute__((always_inline)) {
        const int row = run_row(a.runs, t * WT, WT);
        if (row < 0) return;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int x = 0; x < TB; ++x) {
                if constexpr (bools) mask_bool_words<1>(a.mask, b, my_hq[qt], my_l[qt], row + 16 * x + 4 * g, raw[qt][x]);
                else if constexpr (ARR == 2) mask_add_words<4>(a.mask, b, my_hq[qt], my_l[qt], row + 16 * x + 4 * g, raw[qt][x]);
            }
    };
    auto mask_bits = [&](int t) __attribute__((always_inline)) -> uint32_t {
        const bool whole = run_row(a.runs, t * WT, WT) >= 0;
        uint32_t bits = 0;
#pragma unroll
        for (int x = 0; x < TB; ++x)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int slot = t * WT + 16 * x + 4 * g + j;
                const int row = whole ? 0 : slot < a.slots ? slot_to_row(a.runs, slot) : -1;
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    float add;
                    const bool keep = whole ? ((raw[qt][x][0] >> (8 * j)) & 0xffu) != 0u
                                            : row >= 0 && row < a.T && mask_keep(a.mask, b, my_hq[qt], my_l[qt], row, a.L, a.T, add);
                    bits |= keep ? 1u << ((qt * TB + x) * 4 + j) : 0u;
                }
            }
        return bits;
    };
    // the first of this wavefront's tiles from t on (its elements are there) that a row sees
    auto seen_from = [&](int t, uint32_t &bits) __attribute__((always_inline)) -> int {
        bits = t < te ? mask_bits(t) : 0u;
        while (t < te && !__any(bits != 0u)) {
            t += MW;
            // (unseen tiles come in rows: as many as sixteen words hold are asked for at once)
            constexpr int U = 16 / (QT * TB);
            uint32_t w[U][QT][TB][1];
            bool known[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = t + u * MW, row = c < te ? run_row(a.runs, c * WT, WT) : -1;
                known[u] = row >= 0;
                if (row < 0) continue;
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                    for (int x = 0; x < TB; ++x) mask_bool_words<1>(a.mask, b, my_hq[qt], my_l[qt], row + 16 * x + 4 * g, w[u][qt][x]);
            }
            int unseen = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                uint32_t any = 0;
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                    for (int x = 0; x < TB; ++x) any |= known[u] ? w[u][qt][x][0] : 0u;
                if (unseen == u && known[u] && !__any(any != 0u)) unseen = u + 1;
            }
            t += unseen * MW;
            if (t < te) {
                mask_fetch(t);
                bits = mask_bits(t);
            }
        }
        return t;
    };
    int t = first;
    uint32_t bits = 0, next_bits = 0;
    if constexpr (bools) {
        if (t < te) mask_fetch(t);
        t = seen_from(t, bits);
    }
    if (t < te) {  // wave-uniform
        load_k(t);
        if (ARR && t + (bools ? MW : 0) < te) mask_fetch(t + (bools ? MW : 0));
        load_v(t);
    }
    if constexpr (ROT) {
        step.turn(a.turn, bh, R, rot_s);
        __syncthreads();
        const float *qr = rot_s + min(row0 + col, R - 1) * DK + 4 * g;
        if constexpr (QL) {
            for (int s = wave; s < NS; s += MW) q_s[s * 64 + lane] = *reinterpret_cast<const f4 *>(qr + 16 * s);
            __syncthreads();
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) qop[0][s] = *reinterpret_cast<const f4 *>(qr + 16 * s);
        }
    }
    if constexpr (STEP) {
        if (own) {
            PageCursor page = kpage;
            write_row(page.at(st, a.new_slot));
            if (a.new_slot / WT != first) {  // the row's tile is still to be read
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            } else {
                const int tn = a.new_slot % WT;
#pragma unroll
                for (int x = 0; x < TB; ++x) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) kreg[x][s] = x == tn >> 4 && col == (tn & 15) ? own_k[s] : kreg[x][s];
#pragma unroll
                    for (int c = 0; c < NCT; ++c)
#pragma unroll
                        for (int j = 0; j < 4; ++j) vreg[x][c][j] = 16 * x + 4 * g + j == tn ? own_v[c] : vreg[x][c][j];
                }
            }
        }
    }
    while (t < te) {
        int next = t + MW;
        f4 s[QT][TB];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int x = 0; x < TB; ++x) s[qt][x] = f4{0.f, 0.f, 0.f, 0.f};
        f4 q[QT], qn[QT];
#pragma unroll
        for (int qt = 0; qt < (QL ? QT : 0); ++qt) qn[qt] = q_s[qt * NS * 64 + lane];
#pragma unroll
        for (int e = 0; e < NS; ++e) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                if constexpr (QL) {
                    q[qt] = qn[qt];
                    qn[qt] = q_s[(qt * NS + min(e + 1, NS - 1)) * 64 + lane];
                } else {
                    q[qt] = qop[qt][e];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int x = 0; x < TB; ++x)
#pragma unroll
                    for (int qt = 0; qt < QT; ++qt) s[qt][x] = mfma4(kreg[x][e][j], q[qt][j], s[qt][x]);
            if constexpr (QL) __builtin_amdgcn_sched_barrier(0);  // (one step's queries ahead, not all of them: registers)
        }
        if constexpr (bools) next = seen_from(next, next_bits);
        if (!BRANCH || next < te) load_k(next < te ? next : t);
        const int slot0 = t * WT;
        const bool whole = ARR == 2 && run_row(a.runs, slot0, WT) >= 0;  // wave-uniform
        const bool full = ident && slot0 >= keys.full_lo && slot0 + WT - 1 <= keys.full_hi;  // wave-uniform
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
            for (int x = 0; x < TB; ++x) s[qt][x] *= a.scale;
            if constexpr (bools) {
#pragma unroll
                for (int x = 0; x < TB; ++x)
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[qt][x][j] = (bits >> ((qt * TB + x) * 4 + j)) & 1u ? s[qt][x][j] : -INFINITY;
            } else if (whole) {
#pragma unroll
                for (int x = 0; x < TB; ++x) {
                    if constexpr (ARR == 2) {
                        float add[4];
                        mask_add_floats<4>(a.mask, raw[qt][x], add);
#pragma unroll
                        for (int j = 0; j < 4; ++j) s[qt][x][j] += add[j];
                    }
                }
            } else if (ARR == 0 && ONE && rb.one && ident) {  // one token: every row sees keys.lo to keys.hi
                if (!full) {
#pragma unroll
                    for (int x = 0; x < TB; ++x)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int row = slot0 + 16 * x + 4 * g + j;
                            s[qt][x][j] = row >= keys.lo && row <= keys.hi ? s[qt][x][j] : -INFINITY;
                        }
                }
            } else if (!full) {
#pragma unroll
                for (int x = 0; x < TB; ++x)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int slot = slot0 + 16 * x + 4 * g + j;
                        const int row = ident ? slot : slot < a.slots ? slot_to_row(a.runs, slot) : -1;
                        float add = 0.f;
                        const bool keep = row >= 0 && row < a.T && mask_keep(a.mask, b, my_hq[qt], my_l[qt], row, a.L, a.T, add);
                        s[qt][x][j] = keep ? s[qt][x][j] + add : -INFINITY;
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int x = 0; x < TB; ++x)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[qt][x][j] = fmaxf(s[qt][x][j], -INFINITY);  // (a score that is NaN weighs nothing)
                    mx = fmaxf(mx, s[qt][x][j]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            // (the reference is raised only by more than 3, so that the accumulators are rarely touched after the first tiles)
            const bool raise = mx - m_run[qt] > 3.f || (m_run[qt] == -INFINITY && mx > -INFINITY);
            if (__any(raise)) {
                const float m_new = raise ? mx : m_run[qt];
                const float alpha = raise ? expf(m_run[qt] - m_new) : 1.f;
                l_run[qt] *= alpha;
#pragma unroll
                for (int c = 0; c < NCT; ++c) acc[qt][c] *= alpha;
                m_run[qt] = m_new;
            }
            const float m_use = m_run[qt] > -INFINITY ? m_run[qt] : 0.f;
#pragma unroll
            for (int x = 0; x < TB; ++x)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float p = expf(s[qt][x][j] - m_use);
                    s[qt][x][j] = p;
                    l_run[qt] += p;
                }
        }
#pragma unroll
        for (int x = 0; x < TB; ++x)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < NCT; ++c)
#pragma unroll
                    for (int qt = 0; qt < QT; ++qt) acc[qt][c] = mfma4(vreg[x][c][j], s[qt][x][j], acc[qt][c]);
        if (ARR && next + (bools ? MW : 0) < te) mask_fetch(next + (bools ? MW : 0));
        if (!BRANCH || next < te) load_v(next < te ? next : t);
        t = next;
        bits = next_bits;
    }

    // ---- the four wavefronts' states: each scales its own to the common maximum, then adds up a quarter of the columns ----
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        l_run[qt] += __shfl_xor(l_run[qt], 16);
        l_run[qt] += __shfl_xor(l_run[qt], 32);
        if (g == 0) {
            max_s[wave][qt][col] = m_run[qt];
            sum_s[wave][qt][col] = l_run[qt];
        }
    }
    __syncthreads();
    float M[QT], L[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        M[qt] = max_s[0][qt][col];
#pragma unroll
        for (int w = 1; w < MW; ++w) M[qt] = fmaxf(M[qt], max_s[w][qt][col]);
        L[qt] = 0.f;
#pragma unroll
        for (int w = 0; w < MW; ++w) {
            const float mw = max_s[w][qt][col];
            if (mw > -INFINITY) L[qt] += sum_s[w][qt][col] * expf(mw - M[qt]);
        }
        const float f = m_run[qt] > -INFINITY ? expf(m_run[qt] - M[qt]) : 0.f;
#pragma unroll
        for (int c = 0; c < NCT; ++c) acc_s[((wave * QT + qt) * NCT + c) * 64 + lane] = acc[qt][c] * f;
    }
    __syncthreads();
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int rr = row0 + 16 * qt + col;
        if (rr >= R) continue;
        float *dst = nparts == 1 ? reinterpret_cast<float *>(a.out) + ((size_t)(b * a.Hq + my_hq[qt]) * a.L + my_l[qt]) * DV
                                 : a.workspace + ((size_t)(bh * nparts + part) * R + rr) * (DV + 2);
        for (int c = wave; c < NCT; c += MW) {
            f4 v = acc_s[(qt * NCT + c) * 64 + lane];
#pragma unroll
            for (int w = 1; w < MW; ++w) v += acc_s[((w * QT + qt) * NCT + c) * 64 + lane];
            if (nparts == 1) v = L[qt] > 0.f ? v / L[qt] : f4{0.f, 0.f, 0.f, 0.f};
            float *d = dst + 16 * c + 4 * g;  // (partials: rows of DV + 2 floats, 8-byte aligned; outputs: as their elements are)
            *reinterpret_cast<kv_out2f *>(d) = kv_out2f{v.x, v.y};
            *reinterpret_cast<kv_out2f *>(d + 2) = kv_out2f{v.z, v.w};
        }
        if (nparts > 1 && wave == 0 && g == 0) {
            dst[DV] = M[qt];
            dst[DV + 1] = L[qt];
        }
    }
}

struct PlanF32 {
    int qt, tb, row_blocks, tiles, nparts;
};

PlanF32 plan_f32(const AttendArgs &a) {
    PlanF32 p;
    const int R = (a.Hq / a.Hkv) * a.L;
    p.qt = R <= 16 ? 1 : query_tiles(a.st.Dk);
    p.row_blocks = (R + 16 * p.qt - 1) / (16 * p.qt);
    // A few rows over so few keys that wide tiles would leave wavefronts of the resident workgroups (two per CU) without one:
    // tiles of one token block (one sequence of 1500 keys, 4 kv heads of 64: the kernel 11.0 us with tiles of 64 tokens, of
    // which each workgroup has one).
    p.tb = token_blocks(a.st.Dk, p.qt);
    if (p.qt == 1 && (long)((a.slots + 16 * p.tb - 1) / (16 * p.tb)) * a.st.BH < 512 * MW) p.tb = 1;
    const int wt = 16 * p.tb;
    p.tiles = (a.slots + wt - 1) / wt;
    static const int target = measure_knob("KVHIP_F32_TARGET", 512), least = measure_knob("KVHIP_F32_LEAST", 2);  // (timing builds only)
    const long wgs = (long)p.row_blocks * a.st.BH;
    int n = (int)std::max(1L, std::min<long>(target / std::max(1L, wgs), p.tiles / least));
    n = std::min(n, 32);  // (a merge of 64 parts takes as long as the halves save: 8192 keys, 8 kv heads of 128: 27.6 against 20.7 us)
    const size_t per_part = (size_t)a.st.BH * R * (a.st.Dv + 2) * sizeof(float);
    while (n > 1 && a.workspace_cap && per_part * n > a.workspace_cap) --n;
    p.nparts = n;
    return p;
}

template <int DK, int DV, int QT, int TB>
hipError_t launch_instance(const AttendArgs &a, const PlanF32 &p, hipStream_t s) {
    const dim3 grid(p.row_blocks, a.st.BH, p.nparts), block(256);
    const size_t lds = MW * QT * (DV / 16) * 64 * sizeof(f4);
    const int r = a.Hq / a.Hkv;
    if constexpr (QT == 1) {
        if (a.new_k && a.rope) {
            hipLaunchKernelGGL((attend_f32_kernel<DK, DV, 1, TB, 0, true, true>), grid, block, lds, s, AttendStepArgs(a), r, p.tiles, p.nparts);
            return hipGetLastError();
        }
        if ((DK <= 128 || a.L == 1) && a.mask.mode != KVHIP_MASK_ARRAY) {
            hipLaunchKernelGGL((attend_f32_kernel<DK, DV, 1, TB, 0, false, true>), grid, block, lds, s, a, r, p.tiles, p.nparts);
            return hipGetLastError();
        }
    }
    if (a.mask.mode == KVHIP_MASK_ARRAY) {
        if (a.mask.dtype == KVHIP_BOOL) hipLaunchKernelGGL((attend_f32_kernel<DK, DV, QT, TB, 1, false, false>), grid, block, lds, s, a, r, p.tiles, p.nparts);
        else hipLaunchKernelGGL((attend_f32_kernel<DK, DV, QT, TB, 2, false, false>), grid, block, lds, s, a, r, p.tiles, p.nparts);
    } else if constexpr (QT > 1 || DK > 128) {
        hipLaunchKernelGGL((attend_f32_kernel<DK, DV, QT, TB, 0, false, false>), grid, block, lds, s, a, r, p.tiles, p.nparts);
    }
    return hipGetLastError();
}

template <int DK, int DV>
hipError_t launch_sizes(const AttendArgs &a, const PlanF32 &p, hipStream_t s) {
    if constexpr (token_blocks(DK, 1) != 1) {
        if (p.tb == 1 && p.qt == 1) return launch_instance<DK, DV, 1, 1>(a, p, s);
    }
    if (p.qt == 1) return launch_instance<DK, DV, 1, token_blocks(DK, 1)>(a, p, s);
    return launch_instance<DK, DV, query_tiles(DK), token_blocks(DK, query_tiles(DK))>(a, p, s);
}

}  // namespace

bool attend_f32_supported(const AttendArgs &a) {
    const Store &s = a.st;
    if (s.bits != 0 || s.dtype != KVHIP_F32 || s.BH > 65535) return false;
    // Few query rows over many pairs of head size 256 and enough keys are bound by HBM, where the vector-ALU kernel's 1 KB
    // loads are the better ones (B8, 8 kv heads, 8192 keys, one token: 185 us against 201; B4, 4 kv heads, 4096 keys: 36.2
    // against 37.0; but one sequence, 8 kv heads, 8192 keys: 40.6 against 31).
    if (s.Dk == 256 && s.BH >= 16 && (size_t)s.BH * a.T >= 65536 && (a.Hq / a.Hkv) * a.L <= 8) return false;
    // So are one to four rows over many pairs of the smaller sizes, without a mask that leaves tiles out, in the ranges
    // where they measured 3 to 25 % ahead (vector ALUs / here; outside them this kernel is equal or ahead).  One row: 67 MB
    // of 128 pairs D 64 21.9 / 24.5 us, D 96 101 MB 25.7 / 28.4, D 128 134 MB 30.8 / 35.2 and 1074 MB 176 / 198, 256 pairs of
    // 256 keys 20.1 / 26.2, but D 64 537 MB 112 / 101, 16 pairs 34 MB 16.5 / 15.3.  Four rows: D 128 134 MB 32.0 / 35.8, 1074 MB
    // 182 / 199, but 32 pairs 537 MB 106 / 101, D 96 201 MB 42.0 / 42.0.
    const int R = (a.Hq / a.Hkv) * a.L;
    const size_t mb = (size_t)s.BH * a.T * (s.Dk + s.Dv) * 4 >> 20;
    if (s.Dk == s.Dv && a.mask.mode <= KVHIP_MASK_CAUSAL) {
        const bool many = s.BH >= 256;
        if (R == 1 && s.Dk <= 128 && s.BH >= 16 && mb >= (many ? 32 : 64) && (s.Dk == 128 || mb < 256)) return false;
        if (R <= 4 && s.Dk == 64 && s.BH >= 32 && mb >= (many ? 32 : 64) && mb < 256) return false;
        if (R <= 4 && s.Dk == 128 && s.BH >= 32 && mb >= (many ? 64 : 128) && (s.BH >= 64 || mb < 256)) return false;
        if (R == 1 && s.Dk == 256 && s.BH >= 128 && mb >= 64) return false;
    }
    return (s.Dk == 192 && s.Dv == 128) || (s.Dk == s.Dv && (s.Dk == 64 || s.Dk == 96 || s.Dk == 128 || s.Dk == 256));
}

size_t attend_f32_workspace(const AttendArgs &a) {
    const PlanF32 p = plan_f32(a);
    return p.nparts == 1 ? 0 : (size_t)a.st.BH * p.nparts * (a.Hq / a.Hkv) * a.L * (a.st.Dv + 2) * sizeof(float);
}

hipError_t launch_attend_f32(const AttendArgs &a, hipStream_t s) {
    const PlanF32 p = plan_f32(a);
    profile_mark(s, true);
    hipError_t e;
    if (a.st.Dk == 192) e = launch_sizes<192, 128>(a, p, s);
    else if (a.st.Dk == 64) e = launch_sizes<64, 64>(a, p, s);
    else if (a.st.Dk == 96) e = launch_sizes<96, 96>(a, p, s);
    else if (a.st.Dk == 128) e = launch_sizes<128, 128>(a, p, s);
    else e = launch_sizes<256, 256>(a, p, s);
    profile_mark(s, false);
    if (e != hipSuccess || p.nparts == 1) return e;
    return launch_merge_valu(a, p.nparts, s);
}

}  // namespace kvhip
