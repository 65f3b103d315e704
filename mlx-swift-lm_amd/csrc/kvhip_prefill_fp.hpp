// What the chunked-prefill kernels for full-precision caches share: operands, requests from global memory into LDS, the
// order of the workgroups and the key tiles that one visits.
#pragma once
#include "kvhip_mask.hpp"

namespace kvhip {
namespace prefill_fp {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));


// 16 bytes per lane from global memory straight into LDS: lane i's land at `lds_wave_base` + 16 i
// (the base is the same for the whole wavefront).  Written as assembly, with the waits for it placed
// by hand (s_waitcnt vmcnt): the compiler's own bookkeeping of such loads makes every LDS read that
// follows one wait for all vector-memory operations in flight, register loads included, wherever it
// cannot prove on every path which buffer the load fills.  Its waits for its own loads stay correct:
// vector-memory operations complete in order, so an operation it does not count only makes a wait
// stricter.
// INVARIANT for anyone who edits this kernel: (1) an iteration ends with vmcnt(0) and a barrier before
// any wavefront reads the buffer the loads fill, and every wavefront of the workgroup runs the same
// iterations with the same requests (which variant of an iteration it runs may differ); (2)
// vector-memory operations of one wavefront complete in order on this hardware -- the compiler's own
// waits for register loads rely on that when an uncounted LDS load sits between them.
// (address = wave-uniform 64-bit `base` in scalar registers + the lane's unsigned 32-bit byte offset)
__device__ __forceinline__ void load_to_lds(const char *base, uint32_t lane_off, const void *lds_wave_base) {
    // (the low half of a flat address inside the LDS aperture is the LDS address itself)
    const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds_wave_base);
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    // (readfirstlane returns a signed int: without the casts the low half would be sign-extended over the high one)
    const uint32_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint64_t sb = ((uint64_t)b_hi << 32) | (uint64_t)b_lo;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(sb), "s"(lds) : "memory", "m0");
}
union Op8 {
    h8 h;
    b8 b;
    u4 v;
};


constexpr int BN = 32;  // key slots per tile
constexpr float RAISE = 8.f;  // log2 units

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Workgroups go to the 8 XCDs round-robin by linear id, and each XCD has its own L2.  All
// query blocks of one (batch, kv-head) pair re-read that pair's K and V, so they are given
// ids of the same residue: a pair's tiles then stay hot in one L2 instead of missing in all.
struct WorkItem {
    int block, bh, split;  // block of query rows, (batch, kv head) pair, key-range part
};
template <int MM> __device__ __forceinline__ WorkItem work_item(const AttendArgs &a, int nblk, int nsplit) {
    WorkItem w;
    const int id = blockIdx.x;
    const int BH = a.st.BH;
    if ((BH & 7) == 0) {
        const int xcd = id & 7;
        int j = id >> 3;
        // A grid of exactly two workgroups per CU is resident all at once and gets no balancing from the
        // order of the ids.  Under a causal or window mask the two workgroups of a CU -- 32 apart among the
        // 64 of their XCD -- then take a long and a short query block: the second 32 count backwards.
        if (MM == 1 && gridDim.x == 512 && (j & 32)) j = 95 - j;
        const int per_pair = nblk * nsplit;
        const int h_local = j / per_pair, rem = j - h_local * per_pair;
        w.bh = h_local * 8 + xcd;
        w.split = rem / nblk;
        w.block = rem - w.split * nblk;
    } else {
        w.block = id % nblk;
        const int t = id / nblk;
        w.bh = t % BH;
        w.split = t / BH;
    }
    // Under a causal or window mask the later query blocks see more keys: they are given the lower
    // workgroup ids, which the hardware starts first, so that the launch does not end on its longest blocks.
    if (MM == 1) w.block = nblk - 1 - w.block;
    return w;
}

// The tiles to visit, in slot order, as up to NSEG segments; position v of the visiting order is tile
// vt_of(v).  With slots in presented order that is the one range found above.  A ring presented
// through a run table keeps its rows in rotated order, so the rows no query of this block can see
// (older than the window, newer than the block) lie somewhere inside the slot range: thread 0 maps
// the visible row range through every run to slot tiles, sorts and merges them (a few dozen scalar
// steps, once per workgroup), and whole tiles of invisible rows are never requested -- 14 of 144
// tiles for a 512-row chunk over a 4096-row window.
constexpr int NSEG = 4;
struct Visit {
    int keep_lo, keep_hi;          // the rows that all of the workgroup's queries keep
    int start[NSEG], count[NSEG];  // the tiles to visit
    int lo, hi;                    // this part of the visiting order
    __device__ __forceinline__ int tile(int v) const {
        int t = start[0] + v, rem = v - count[0];
#pragma unroll
        for (int k = 1; k < NSEG; ++k) {
            if (rem >= 0) t = start[k] + rem;
            rem -= count[k];
        }
        return t;
    }
};
struct VisitShared {
    int lo[MAXRUNS], hi[MAXRUNS], n;
};
template <int BM, int MM, bool IDENT>
__device__ __forceinline__ Visit visit_plan(const AttendArgs &a, const SymMask &sym, int block, int R, int split, int nsplit, VisitShared &sh) {
    Visit w;
    w.keep_lo = 0;
    w.keep_hi = -1;
    int tile_lo = 0, tile_hi = (a.slots + BN - 1) / BN;
    {
        const int i_first = block * BM, i_last = min(R, i_first + BM) - 1;
        const bool spans = (i_first / a.L) != (i_last / a.L);
        const int l_min = spans ? 0 : i_first % a.L, l_max = spans ? a.L - 1 : i_last % a.L;
        if (MM != 2) {
            w.keep_hi = a.T - 1;
            if (MM == 1) {
                if (sym.mode == KVHIP_MASK_CAUSAL) {
                    w.keep_hi = a.T - a.L + l_min;
                } else {
                    w.keep_lo = sym.pad_b;
                    w.keep_hi = min(sym.offset + l_min, sym.len_b - 1);
                    if (sym.window > 0) w.keep_lo = max(w.keep_lo, sym.offset + l_max - sym.window + 1);
                }
                w.keep_hi = min(w.keep_hi, a.T - 1);
            }
        }
        if (IDENT) {  // slots are presented rows: tiles outside a symbolic mask are skipped
            if (a.mask.mode == KVHIP_MASK_CAUSAL) {
                tile_hi = min(tile_hi, (a.T - a.L + l_max) / BN + 1);
            } else if (a.mask.mode == KVHIP_MASK_WINDOW) {
                tile_hi = min(tile_hi, (a.mask.offset + l_max) / BN + 1);
                if (a.mask.window > 0) tile_lo = max(0, (a.mask.offset + l_min - a.mask.window + 1) / BN);
            }
            tile_hi = min(tile_hi, (a.T + BN - 1) / BN);
        }
    }
#pragma unroll
    for (int k = 0; k < NSEG; ++k) w.start[k] = w.count[k] = 0;
    w.start[0] = tile_lo;
    w.count[0] = max(tile_hi - tile_lo, 0);
    if constexpr (!IDENT && MM == 1) {
        if (threadIdx.x == 0) {
            const int i_first = block * BM, i_last = min(R, i_first + BM) - 1;
            const bool spans = (i_first / a.L) != (i_last / a.L);
            const int l_min = spans ? 0 : i_first % a.L, l_max = spans ? a.L - 1 : i_last % a.L;
            int vis_lo = 0, vis_hi = a.T - a.L + l_max;  // rows some query of the block may see
            if (sym.mode != KVHIP_MASK_CAUSAL) {
                vis_lo = sym.pad_b;
                vis_hi = min(sym.offset + l_max, sym.len_b - 1);
                if (sym.window > 0) vis_lo = max(vis_lo, sym.offset + l_min - sym.window + 1);
            }
            vis_lo = max(vis_lo, 0);
            vis_hi = min(vis_hi, a.T - 1);
            int ns = 0;
#pragma unroll
            for (int i = 0; i < MAXRUNS; ++i) {
                if (i < a.runs.n) {
                    const int r_lo = max(vis_lo, a.runs.row0[i]), r_hi = min(vis_hi, a.runs.row0[i] + a.runs.len[i] - 1);
                    if (r_lo <= r_hi) {
                        const int t_lo = (a.runs.phys0[i] + r_lo - a.runs.row0[i]) / BN;
                        const int t_hi = (a.runs.phys0[i] + r_hi - a.runs.row0[i]) / BN;
                        int pos = ns;  // insertion by first tile
                        while (pos > 0 && sh.lo[pos - 1] > t_lo) {
                            sh.lo[pos] = sh.lo[pos - 1];
                            sh.hi[pos] = sh.hi[pos - 1];
                            --pos;
                        }
                        sh.lo[pos] = t_lo;
                        sh.hi[pos] = t_hi;
                        ++ns;
                    }
                }
            }
            int m = 0;  // merge what overlaps or touches
            for (int i = 0; i < ns; ++i) {
                if (m > 0 && sh.lo[i] <= sh.hi[m - 1] + 1) {
                    sh.hi[m - 1] = max(sh.hi[m - 1], sh.hi[i]);
                } else {
                    sh.lo[m] = sh.lo[i];
                    sh.hi[m] = sh.hi[i];
                    ++m;
                }
            }
            if (m > NSEG) {  // more pieces than are kept: one range over all of them (nothing wrong, nothing skipped)
                sh.hi[0] = sh.hi[m - 1];
                m = 1;
            }
            sh.n = m;
        }
        __syncthreads();
        const int m = __builtin_amdgcn_readfirstlane(sh.n);
#pragma unroll
        for (int k = 0; k < NSEG; ++k) {
            const int lo = k < m ? __builtin_amdgcn_readfirstlane(sh.lo[k]) : 0;
            const int hi = k < m ? __builtin_amdgcn_readfirstlane(sh.hi[k]) : -1;
            w.start[k] = lo;
            w.count[k] = hi - lo + 1;
        }
    }
    w.lo = w.hi = 0;
#pragma unroll
    for (int k = 0; k < NSEG; ++k) w.hi += w.count[k];
    // optional split of the visiting order (small grids): each part leaves an
    // unnormalised partial per query row, merged by the decode path's combine kernel
    if (nsplit > 1) {
        const int span = (w.hi + nsplit - 1) / nsplit;
        w.lo = split * span;
        w.hi = min(w.hi, w.lo + span);
    }
    return w;
}

}  // namespace prefill_fp
}  // namespace kvhip
