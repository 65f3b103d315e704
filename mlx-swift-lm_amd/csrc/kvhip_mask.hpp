// Mask evaluation shared by the attention kernels.
#pragma once
#include "kvhip_device.hpp"
#include "kvhip_wave.hpp"

namespace kvhip {

// Decides whether query row l (of L) of batch b / query head hq may see presented
// key row j (of T).  `add` receives the additive term of a float array mask.
__device__ __forceinline__ bool mask_keep(const MaskDev &m, int b, int hq, int l, int j, int L, int T,
                                          float &add) {
    add = 0.0f;
    switch (m.mode) {
        case KVHIP_MASK_CAUSAL:
            return j <= T - L + l;
        case KVHIP_MASK_ARRAY: {
            const size_t i = (size_t)(b * m.sb + hq * m.sh + l * m.sl) + j;
            if (m.dtype == KVHIP_BOOL) return reinterpret_cast<const uint8_t *>(m.data)[i] != 0;
            if (m.dtype == KVHIP_F16) add = Elem<0>::load(m.data, i);
            else if (m.dtype == KVHIP_BF16) add = Elem<1>::load(m.data, i);
            else add = Elem<2>::load(m.data, i);
            return true;
        }
        case KVHIP_MASK_WINDOW: {
            const int li = m.offset + l;
            bool keep = li >= j;
            if (m.window > 0) keep = keep && (li < j + m.window);
            if (m.lengths) keep = keep && (j < m.lengths[b]);
            if (m.left_pad) keep = keep && (j >= m.left_pad[b]);
            return keep;
        }
        default:
            return true;
    }
}

// 4 * W consecutive bytes of a boolean array mask: query row l of (b, hq), key rows j0 .. j0 + 4 W - 1
// (all below T; the address need not be aligned: global loads take any byte address).  One
// load in place of 4 W byte loads per lane.
template <int W>
__device__ __forceinline__ void mask_bool_words(const MaskDev &m, int b, int hq, int l, int j0, uint32_t (&w)[W]) {
    const uint8_t *p = reinterpret_cast<const uint8_t *>(m.data) + (size_t)(b * m.sb + hq * m.sh + l * m.sl) + j0;
    struct __attribute__((packed, aligned(1))) Raw {
        uint32_t v[W];
    };
    const Raw raw = *reinterpret_cast<const Raw *>(p);
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = raw.v[i];
}

// The presented row of `slot0` when the slots slot0 .. slot0 + n - 1 lie in one run (wave-uniform); -1 otherwise.
__device__ __forceinline__ int run_row(const Runs &r, int slot0, int n) {
    int row = -1;
#pragma unroll
    for (int i = 0; i < MAXRUNS; ++i)
        if (i < r.n && slot0 >= r.phys0[i] && slot0 + n <= r.phys0[i] + r.len[i]) row = r.row0[i] + slot0 - r.phys0[i];
    return row;
}
// Elements row .. row + N - 1 (all presented) of an additive array mask for query row l of (b, hq), as they lie in memory
// (a wide load, which can be requested well before the scores that the elements belong to), and as floats.
template <int N> __device__ __forceinline__ void mask_add_words(const MaskDev &m, int b, int hq, int l, int row, uint32_t (&w)[N]) {
    struct __attribute__((packed, aligned(1))) Raw32 {
        uint32_t v[N];
    };
    struct __attribute__((packed, aligned(1))) Raw16 {
        uint32_t v[N / 2];
    };
    const size_t i = (size_t)(b * m.sb + hq * m.sh + l * m.sl) + row;
    if (m.dtype == KVHIP_F32) {
        const Raw32 x = *reinterpret_cast<const Raw32 *>(reinterpret_cast<const char *>(m.data) + 4 * i);
#pragma unroll
        for (int k = 0; k < N; ++k) w[k] = x.v[k];
    } else {
        const Raw16 x = *reinterpret_cast<const Raw16 *>(reinterpret_cast<const char *>(m.data) + 2 * i);
#pragma unroll
        for (int k = 0; k < N; ++k) w[k] = k < N / 2 ? x.v[k % (N / 2)] : 0u;
    }
}
template <int N> __device__ __forceinline__ void mask_add_floats(const MaskDev &m, const uint32_t (&w)[N], float (&add)[N]) {
    const bool f32 = m.dtype == KVHIP_F32, bf16 = m.dtype == KVHIP_BF16;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const uint32_t whole = w[j], half = w[j >> 1] >> (16 * (j & 1));
        const float narrow = bf16 ? __uint_as_float(half << 16) : __half2float(__ushort_as_half((unsigned short)half));
        add[j] = f32 ? __uint_as_float(whole) : narrow;
    }
}

// Index-only masks (causal, window with optional per-batch bounds) with the per-batch
// bounds already in registers: no memory access, so kernels can keep loads in flight.
struct SymMask {
    int mode, offset, window, len_b, pad_b, T, L;
};
__device__ __forceinline__ SymMask sym_mask_init(const MaskDev &m, int b, int L, int T) {
    SymMask s;
    s.mode = m.mode;
    s.offset = m.offset;
    s.window = m.window;
    s.len_b = (m.mode == KVHIP_MASK_WINDOW && m.lengths) ? m.lengths[b] : 0x7fffffff;
    s.pad_b = (m.mode == KVHIP_MASK_WINDOW && m.left_pad) ? m.left_pad[b] : 0;
    s.T = T;
    s.L = L;
    return s;
}
// The key rows [lo, hi] that query position l sees (empty if lo > hi): two comparisons a key in the tiles at the edges.
// (Evaluated condition by condition for every key, such a tile took the 16-row kernel as long as two others.)
struct KeyBounds {
    int lo, hi;
    __device__ __forceinline__ bool keep(int j) const { return j >= lo && j <= hi; }
};
// (No branches: a wavefront forms those of four rows and more per group at its start.)
__device__ __forceinline__ KeyBounds sym_mask_bounds(const SymMask &s, int l) {
    const bool causal = s.mode == KVHIP_MASK_CAUSAL;
    const int from = !causal && s.window > 0 ? s.offset - s.window + 1 : -0x40000000, upto = causal ? s.T - s.L : s.offset;
    return KeyBounds{max(causal ? 0 : s.pad_b, from + l), min(causal ? 0x7fffffff : s.len_b - 1, upto + l)};
}

// Inclusive range of key rows any query position l in [0, L) may see under an index-only mask.
__device__ __forceinline__ void sym_mask_row_range(const SymMask &s, int &lo, int &hi) {
    if (s.mode == KVHIP_MASK_CAUSAL) {
        lo = 0;
        hi = s.T - 1;
        return;
    }
    lo = s.pad_b;
    hi = min(s.offset + s.L - 1, s.len_b - 1);
    if (s.window > 0) lo = max(lo, s.offset - s.window + 1);
}

// Whether some query position l in [0, L) sees no key row at all.  The quantized path fills
// masked scores with finfo.min instead of dropping them (KVCache.swift:2396-2447), so such a
// row attends uniformly over ALL presented keys and no key tile may be skipped for it.
__device__ __forceinline__ bool sym_mask_some_row_empty(const SymMask &s) {
    if (s.mode == KVHIP_MASK_CAUSAL) return s.T - s.L < 0;
    // per position l the kept rows are [max(pad, offset + l - window + 1), min(offset + l, len - 1)]:
    // the width is concave in l, so it is smallest at one of the two ends
    for (int e = 0; e < 2; ++e) {
        const int l = e ? s.L - 1 : 0;
        int lo = s.pad_b;
        const int hi = min(s.offset + l, min(s.len_b, s.T) - 1);
        if (s.window > 0) lo = max(lo, s.offset + l - s.window + 1);
        if (lo > hi) return true;
    }
    return false;
}

// Inclusive range of key rows EVERY query position l in [0, L) sees (empty if lo > hi).
__device__ __forceinline__ void sym_mask_full_range(const SymMask &s, int &lo, int &hi) {
    if (s.mode == KVHIP_MASK_CAUSAL) {
        lo = 0;
        hi = s.T - s.L;
        return;
    }
    lo = s.pad_b;
    hi = min(s.offset, s.len_b - 1);
    if (s.window > 0) lo = max(lo, s.offset + s.L - s.window);
}

// Key rows some (lo .. hi) and all (full_lo .. full_hi) of the query positions l0 .. l1 of batch row b see, both
// inclusive, empty if low > high; array masks: every key, and none for certain.
struct KeyRange {
    int lo, hi, full_lo, full_hi;
};
__device__ __forceinline__ KeyRange visible_keys(const MaskDev &m, int b, int L, int T, int l0, int l1) {
    KeyRange k{0, T - 1, 0, T - 1};
    if (m.mode == KVHIP_MASK_CAUSAL) {
        k.hi = min(k.hi, T - L + l1);
        k.full_hi = min(k.full_hi, T - L + l0);
    } else if (m.mode == KVHIP_MASK_WINDOW) {
        const SymMask s = sym_mask_init(m, b, L, T);
        k.lo = k.full_lo = max(0, s.pad_b);
        if (s.window > 0) {
            k.lo = max(k.lo, s.offset + l0 - s.window + 1);
            k.full_lo = max(k.full_lo, s.offset + l1 - s.window + 1);
        }
        k.hi = min(k.hi, min(s.offset + l1, s.len_b - 1));
        k.full_hi = min(k.full_hi, min(s.offset + l0, s.len_b - 1));
    } else if (m.mode == KVHIP_MASK_ARRAY) {
        k.full_hi = -1;
    }
    return k;
}

// The workgroup of a grid (row blocks, BH, parts): its row block, pair and part, and which head and position a query row is.
// No division where a step needs none: a dozen of them stood between a step's start and its first request (1.5 us of the
// 2.7 of a step of head size 512).
struct RowBlock {
    int block, bh, part, b, h;
    int L;
    bool one;  // one new token: a row is a head
    __device__ __forceinline__ RowBlock(const AttendArgs &a) : block(0), bh(blockIdx.y), part(blockIdx.z), L(a.L), one(a.L == 1) {
        if (gridDim.x > 1) {
            // (the row blocks of one kv head and part run on one XCD and share its L2: see attend_valu_kernel)
            int lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
            const int total = gridDim.x * gridDim.y * gridDim.z;
            if ((total & 7) == 0) lin = (lin & 7) * (total >> 3) + (lin >> 3);
            const int rest = lin / gridDim.x;
            block = lin - rest * gridDim.x;
            part = rest / gridDim.y;
            bh = rest - part * gridDim.y;
        }
        b = a.B == 1 ? 0 : bh / a.Hkv;
        h = bh - b * a.Hkv;
    }
    __device__ __forceinline__ int head(int row) const { return one ? row : row / L; }
    __device__ __forceinline__ int pos(int row) const { return one ? 0 : row % L; }
};

// ---- the spans of a ragged batch -----------------------------------------------------------------------------------
// The 64-token tiles batch row `b` sees, [lo, hi).  `all_if_empty`: a query position that sees no key averages over every
// one of them (the quantized path), so no tile may be left out for its row.
struct TileRange {
    int lo, hi;
};
__device__ __forceinline__ TileRange visible_tiles(const SymMask &s, int tiles_total, bool all_if_empty) {
    int vis_lo, vis_hi;
    sym_mask_row_range(s, vis_lo, vis_hi);
    TileRange t{max(0, vis_lo) >> 6, min(tiles_total, (min(vis_hi, s.T - 1) >> 6) + 1)};
    if (all_if_empty && sym_mask_some_row_empty(s)) {
        t.lo = 0;
        t.hi = tiles_total;
    }
    return t;
}

// ceil(x / d) for small whole numbers, r = 1 / d (a quotient in float, put right by its remainder)
__device__ __forceinline__ int quotient_up(int x, int d, float r) {
    x += d - 1;
    const int q = (int)((float)x * r), rem = x - q * d;
    return q + (rem >= d ? 1 : rem < 0 ? -1 : 0);
}
// Workgroup `wid` of the nsplit * B that share one kv head's batch rows (2 <= B <= 64, 2 <= nsplit, at most 512 workgroups,
// of `waves` wavefronts each, which take every waves-th tile): all spans have the same length and a row gets as many as its
// keys need, so that the launch lasts as long as the batch's keys do in all and not as its longest row does.  The length is
// the first from an even share on with which the spans go round -- unless the longest row over nsplit spans of its own is
// done as soon, and then every row goes by its own length over up to nsplit spans.  Workgroups without a span are the last.
// Every workgroup works the partition out for itself, a lane to a batch row, and hands on the row's bounds, which are in
// the lanes already (the sums are of small whole numbers, exact in float).  Spans of a row are adjacent:
// first .. first + count - 1; count 0: nothing is left for this workgroup.
// (B16 of 1024 to 16384 keys, 4 new tokens, 8 kv heads of 128 at 4 bits, the kernel 42 us with every row over the same
// number of spans, long rows and short ones paired on the CUs.)
struct RaggedSpan {
    int b, first, count;  // batch row; its spans
    TileRange t;          // this workgroup's tiles
    SymMask sym;          // what the row sees
};
__device__ __forceinline__ RaggedSpan ragged_span(const MaskDev &m, int B, int L, int T, int tiles_total, int nsplit, int waves, int wid, bool all_if_empty) {
    const int lane = threadIdx.x & 63, wgs = nsplit * B;
    const SymMask row = sym_mask_init(m, min(lane, B - 1), L, T);
    const TileRange mine = visible_tiles(row, tiles_total, all_if_empty);
    const int tiles = lane < B ? max(mine.hi - mine.lo, 0) : 0, steps = (tiles + waves - 1) / waves;
    auto lane_of = [](int v, int l) { return __builtin_amdgcn_readlane(v, l); };
    auto end_of = [&](float upto, int l) { return (int)__builtin_bit_cast(float, lane_of(__builtin_bit_cast(int, upto), l)); };
    int len = max(1, quotient_up(steps, nsplit, __builtin_amdgcn_rcpf((float)nsplit)));  // a row's own
    const int most = (int)wave_max((float)len);
    int spans;
    float upto;
    auto share = [&]() {
        spans = lane < B ? max(1, quotient_up(steps, len, __builtin_amdgcn_rcpf((float)len))) : 0;
        upto = wave_scan((float)spans);
        return end_of(upto, 63);
    };
    const int own = len;
    len = max(1, quotient_up((int)wave_sum((float)steps), wgs, __builtin_amdgcn_rcpf((float)wgs)));
    while (len < most && share() > wgs) ++len;
    if (len >= most) {  // wave-uniform
        len = own;
        share();
    }
    const int before = __popcll(__ballot(lane < B && upto <= (float)wid));
    RaggedSpan r;
    r.b = min(before, B - 1);
    r.count = before < B ? lane_of(spans, r.b) : 0;
    r.first = end_of(upto, r.b) - r.count;
    len = lane_of(len, r.b);
    r.t.lo = lane_of(mine.lo, r.b) + (wid - r.first) * len * waves;
    r.t.hi = min(lane_of(mine.hi, r.b), r.t.lo + len * waves);
    r.sym = row;
    r.sym.len_b = lane_of(row.len_b, r.b);
    r.sym.pad_b = lane_of(row.pad_b, r.b);
    return r;
}

// Where such a launch notes, behind its partials, which of them are a pair's: first and count, per (batch row, kv head).
__host__ __device__ __forceinline__ int2 *span_table(float *workspace, int BH, int nsplit, int floats_per_span) {
    return reinterpret_cast<int2 *>(workspace + (size_t)BH * nsplit * floats_per_span);
}

// ---- which batch row a workgroup row takes, for ragged batches ------------------------------------
// (Batches that ragged_span does not take: a single span to a row.)
// Workgroups are started in id order, one per CU and then a second one per CU, so rows v and v + B/2 of a
// launch of 512 workgroups share CUs.  Taking the batch rows in order of their visible length -- the first
// half of the workgroup rows in descending order, the second half in ascending order -- pairs the longest
// row with the shortest on the same CUs, the second longest with the second shortest, and so on, instead of
// whatever the batch order happens to pair.  Every workgroup computes the same permutation (one lane
// per batch row, B <= 64); partial results are still indexed by the batch row itself, so nothing
// downstream changes.
__device__ __forceinline__ int balanced_row(const MaskDev &m, int B, int L, int T, int tiles_total, int v) {
    const int lane = threadIdx.x & 63;
    int tiles = -1;
    if (lane < B) {
        const TileRange t = visible_tiles(sym_mask_init(m, lane, L, T), tiles_total, true);
        tiles = max(t.hi - t.lo, 0);
    }
    int rank = 0;  // rows that come before this lane's: more tiles, or as many and a lower index
    for (int j = 0; j < B; ++j) {
        const int tj = __shfl(tiles, j);
        rank += (tj > tiles || (tj == tiles && j < lane)) ? 1 : 0;
    }
    const int h = (B + 1) / 2;
    const int want = v < h ? v : B - 1 - (v - h);
    const unsigned long long hit = __ballot(lane < B && rank == want);
    return hit ? __ffsll(hit) - 1 : v;
}

}  // namespace kvhip
