// draw_lines on gfx950: segment checkpoints, tile-binned LDS accumulation,
// pixel lists, the deterministic (reference-order) mode, accumulate_lines,
// plans and the adjoint.
//
// Tile path (draw_lines, plans; F frames of H x W, N lines):
//
//  1. k_setup_lines   one lane per line: the line's constants (LineSetup) and
//                     its segment bound; the bound total (the slot count;
//                     an eager draw reads it first only when the previous
//                     call's total is no usable capacity).
//  2. k_walk_lines    one lane per line: replays the reference's walk once,
//                     cutting it into segments of <= SEG long-axis columns
//                     inside the frame.  A segment stores the exact walk
//                     state at its first column (the checkpoint) and the
//                     short-axis pixel range its fills can reach; the walk
//                     counts (segment, tile) items per tile sub-list, one
//                     atomic per run of items into one sub-list.
//  3. k_scan          item offsets per tile sub-list (one host read: the
//                     item total, flags and slot count; plans read nothing).
//  4. k_bin_slots     one lane per segment slot: the per-tile item lists, in
//                     sub-lists of like cost (list_class).
//  5. k_tiles_fast    (cbx_tiles.hip) one workgroup per TILE x TILE pixel tile of
//                     float images, k_tiles of double images and exact values:
//                     each item's walk is resumed from its checkpoint (phase 1,
//                     column records into LDS) and its columns are filled (phase
//                     2) into an LDS tile with LDS atomics (fixed point for float
//                     sums); the tile is flushed to HBM once with a coalesced
//                     read-modify-write.  HBM traffic of the image: one read and
//                     one write per touched tile.
//
// Ordered path (pixel lists, the deterministic mode, accumulate_lines with
// different overlaps): k_segments walks twice (count, then write) so that a
// line's segments are consecutive and lines keep their input order, and
// k_tiles_ordered applies each pixel's terms in ascending line order, the
// single-threaded reference's order.  Float lines of accumulate_lines that no
// other line of their term can touch take the tile path with exact values
// instead (k_term_touch).  The adjoint
// (k_adjoint_fast, k_adjoint_tiles for doubles, k_line_grad) runs on the tile
// path's segments and lists.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstddef>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>

#include "cbx_draw.hpp"

namespace cbx {

// ---------------------------------------------------------------------------
// segment pre-passes
// ---------------------------------------------------------------------------
// Line constants and frame check of line l; false if the line draws nothing.
// kid: the line's profile, kernels[l] when per-line profiles are given.
template <typename T, typename I>
__device__ __forceinline__ bool setup_line(const T *__restrict__ lines, const I *__restrict__ idxs,
                                           const uint8_t *__restrict__ kernels, int kernel, int64_t l,
                                           const Geometry &g, LineSetup<T> &L, int *__restrict__ flags)
{
    int rc = line_setup(lines + 5 * l, L);
    const int kid = kernels ? (int)kernels[l] : kernel;
    L.kid = (int8_t)kid;
    if (kid < K_BIWEIGHT || kid > K_TRIANGULAR) {
        atomicOr(flags, FLAG_KERNEL);
        L.valid = 0;
    }
    int64_t f = idxs ? (int64_t)idxs[l] : ((g.n_frames == 1) ? 0 : l);
    if (f < 0 && g.skip_neg) {
        L.valid = 0;
        f = 0;
    } else if (f < 0 || f >= g.n_frames) {
        atomicOr(flags, FLAG_INDEX);
        L.valid = 0;
    }
    if (rc) {
        atomicOr(flags, rc);
        L.valid = 0;
    }
    L.frame = (int32_t)f;
    L.sub = (int8_t)(L.valid ? list_class(L, kernels != nullptr) : 0);
    return L.valid;
}

__device__ __forceinline__ LineLite line_lite(const LineSetup<float> &L)
{
    const int a = L.axis, b = 1 - a;
    LineLite r;
    r.t[0] = L.t[0];
    r.t[1] = L.t[1];
    r.LL = L.LL;
    r.ea = L.ea;
    r.nlim = L.nlim;
    // A fill visits at most J = nlim / |t_a| + 2 steps from its column, each
    // moving Te by |t_b| and rounding it by at most half an ulp of LL + cap.
    const float J = L.nlim / m_abs(pick(L.t, a)) + 2.0f;
    r.cap = J * (m_abs(pick(L.t, b)) * 1.00001f + L.LL * 2.4e-7f);
    r.meta = a | (pick(L.st, a) > 0 ? FR_SA : 0) | (pick(L.st, b) > 0 ? FR_SB : 0) | (L.safe ? FR_SAFE : 0) |
             ((int)(uint8_t)L.kid << 8);
    return r;
}

// Most segments a line's walk can make: one per SEG-column block of the
// long-axis range [m0, m1] inside the frame (the walk is monotone along the
// long axis and never passes m1).
template <typename T>
__device__ __forceinline__ int segment_bound(const LineSetup<T> &L, const Geometry &g)
{
    if (!L.valid) return 0;
    const int a = L.axis, da = (a == 0) ? g.W : g.H;
    const int c0 = pick(L.m0, a), c1 = pick(L.m1, a);
    const int lo = max(min(c0, c1), 0), hi = min(max(c0, c1), da - 1);
    return (lo > hi) ? 0 : (hi >> g.seg_log) - (lo >> g.seg_log) + 1;
}

// Short-axis pixels from a column's centre that its fills can reach.  A fill of
// j steps has |N_j| >= j |t_a| - |N_0| and stops once |N| / len >= w; at an emitted
// column |N_0| <= max(|N at m0|, |t_a| / 2): every step takes the candidate of
// smallest |N|, and one of them moves N against its sign by at most |t_a|.
// (2^-23 per step: the rounding of the fill's running sums.)
template <typename T>
__device__ __forceinline__ int fill_reach(const LineSetup<T> &L)
{
    const double ta = (double)m_abs(pick(L.t, L.axis));
    const double n0 = (double)m_abs(L.e0[1]), half = 0.50001 * ta;
    const double j = ((double)L.w * (double)L.len + (n0 > half ? n0 : half)) / ta;
    const double r = j * (1.00001 + 1.2e-7 * j) + 1.0;
    return r < 1073741824.0 ? (int)r : 1073741824;   // 2^30: added to a coordinate (below 1e9) it stays an int
}

// Replays line l's walk (bresenham.hpp:352-383) and cuts it into segments of
// <= SEG long-axis columns inside the frame.  For each segment whose fills
// can reach the frame, on_seg(cur, tl) gets the checkpoint (with the reach
// range lo..hi set) and the tile column tl along the long axis.
//
// The steps are a serial chain (each FP32 sum rounds), so the time of a draw of
// few lines is the instructions of one step times the longest line, and the
// loop holds little else: the next |N| is one of the three candidates, both
// coordinates move by selects, one test ends the block.  Emission needs no bookkeeping: every long-axis
// step emits the column it leaves, so a block's emitted columns are its first
// ones, their centres lie between the block's first and last short-axis
// positions and their errors below a bound of the whole line (fill_reach).
// TRACK: the range from the emitted centres and errors themselves, which is a pixel
// narrower for some segments.  The ordered mode takes it, which can sort only so many
// segments of a tile.
// 19 vector instructions per step: the walk of 1000 lines of up to 720 px takes
// 71 us (131 with the bookkeeping in the step and a store ring), of 128 000
// lines of up to 400 px 86 us (126).
template <bool TRACK, typename T, typename OnSeg>
__device__ __forceinline__ void walk_segments(const LineSetup<T> &L, int64_t l, const Geometry &g,
                                              int *__restrict__ flags, OnSeg on_seg)
{
    const int a = L.axis, b = 1 - a;
    const bool ax = a == 1;
    const int da = ax ? g.H : g.W, db = ax ? g.W : g.H;
    const int sa = pick(L.st, a), sb = pick(L.st, b);
    const int R = fill_reach(L);
    int q_first = 0, q_last = 0;   // TRACK: `side` at the block's first and last emitted column,
    T n_most = T(0);               // and the largest |N| at one
    // signed increments along x and y
    const T dx = (L.st[0] > 0) ? L.nv[0] : -L.nv[0], dy = (L.st[1] > 0) ? L.nv[1] : -L.nv[1];
    const T ux = (L.st[0] > 0) ? L.t[0] : -L.t[0], uy = (L.st[1] > 0) ? L.t[1] : -L.t[1];
    T Te = L.e0[0], Ne = L.e0[1];
    int c = pick(L.m0, a), s = pick(L.m0, b);
    int left = (pick(L.m1, a) - c) * sa, side = (pick(L.m1, b) - s) * sb;   // steps to the walk's end along each axis
    wait_vm_loads();

    // steps until k (> 0) long-axis steps are done or `side` (> 0) short-axis
    // steps are left no more; returns the long-axis steps left.  Every step moves
    // along one of the axes at least, so the loop ends.
    auto advance = [&](int k) {
        bool go;
        do {
            const T ex = Ne + dx, ey = Ne + dy, exy = ex + dy;
            const bool yb = m_abs(ey) < m_abs(ex);
            const T m = yb ? ey : ex;
            const bool both = m_abs(exy) < m_abs(m);
            if constexpr (TRACK) {
                const bool em = both | (yb == ax);   // a column is left
                const T an = m_abs(Ne);
                q_first = em ? max(q_first, side) : q_first;
                q_last = em ? side : q_last;
                n_most = (em & (an > n_most)) ? an : n_most;
            }
            Te += (both | !yb) ? ux : T(0);
            Te += (both | yb) ? uy : T(0);
            Ne = both ? exy : m;
            side -= (both | (yb != ax)) ? 1 : 0;
            k -= (both | (yb == ax)) ? 1 : 0;
            go = (k != 0) & (side != 0);
        } while (go);
        return k;
    };

    // columns before the frame (the walk is monotone along the long axis)
    {
        const int k0 = min(max(0, (sa > 0) ? -c : c - (da - 1)), left);
        if (k0 > 0) {
            const int q = side;
            const int k = advance(k0);
            c += sa * k0;
            s += sb * (q - side);
            left = (k != 0) ? 0 : left - k0;
        }
    }
    left = (side > 0) ? min(left, (sa > 0) ? da - c : c + 1) : 0;   // columns inside the frame
    const int seg = g.seg;
    int most = 0;
    Segment<T> cur;
    cur.line = (int32_t)l;
    while (left > 0) {
        // a segment from the current column to the end of its block of SEG
        const int in = c & (seg - 1);
        const int k0 = min((sa > 0) ? seg - in : in + 1, left);
        const int s0 = s, q = side, tl = c >> g.tile_log;
        cur.c[0] = ax ? s : c;
        cur.c[1] = ax ? c : s;
        cur.Te = Te;
        cur.Ne = Ne;
        if constexpr (TRACK) {
            q_first = 0;   // (`side` is positive at every step)
            n_most = T(0);
        }
        const int k = advance(k0);
        most = max(most, q - side);
        s += sb * (q - side);
        c += sa * k0;
        left = (side > 0) ? left - k0 : 0;
        cur.ncols = k0 - k;
        int e0 = s0, e1 = s, r = R;
        if constexpr (TRACK) {
            e0 = s0 + sb * (q - q_first);
            e1 = s0 + sb * (q - q_last);
            // as fill_reach; one of the two pixels is for the rounding of up to 2886 steps
            const double j = ((double)L.w * (double)L.len + (double)n_most) / (double)m_abs(pick(L.t, a));
            const double reach = __builtin_floor(j) + 2.0 + __builtin_floor(1.2e-7 * j * j);
            r = reach < 1073741824.0 ? (int)reach : 1073741824;
        }
        cur.lo = max(min(e0, e1) - r, 0);
        cur.hi = min(max(e0, e1) + r, db - 1);
        if ((cur.ncols > 0) & (cur.lo <= cur.hi)) on_seg(cur, tl);
    }
    // (the tile kernels' replay stops after 4 SEG + 16 steps; a walk takes at
    // most about two per column)
    if (most > 3 * seg + 8) atomicOr(flags, FLAG_STUCK);
}

__device__ __forceinline__ int64_t tile_index(const Geometry &g, int frame, int axis, int tl, int tb)
{
    const int tx = (axis == 0) ? tl : tb, ty = (axis == 0) ? tb : tl;
    return ((int64_t)frame * g.nty + ty) * g.ntx + tx;
}

// Ordered plan (pixel lists, deterministic images, adjoint): segments of a
// line are consecutive and lines are in input order.  Pass 1 (WRITE = false)
// counts segments per line and items per tile; pass 2 writes them at the
// scanned offsets.
template <typename T, typename I, bool WRITE, bool BIN>
__global__ void __launch_bounds__(256)
k_segments(const T *__restrict__ lines, const I *__restrict__ idxs, int kernel, int64_t n_lines, Geometry g,
           LineSetup<T> *__restrict__ setup, int *__restrict__ seg_cnt, int *__restrict__ tile_cnt,
           const int *__restrict__ seg_off, Segment<T> *__restrict__ segs, const int *__restrict__ tile_off,
           int *__restrict__ tile_cur, int *__restrict__ items, int *__restrict__ flags)
{
    int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= n_lines) return;
    LineSetup<T> L;
    if (!WRITE) {
        const bool ok = setup_line(lines, idxs, (const uint8_t *)nullptr, kernel, l, g, L, flags);
        setup[l] = L;
        if (!ok) {
            seg_cnt[l] = 0;
            return;
        }
    } else {
        L = setup[l];
        if (!L.valid) return;
    }
    const int base = WRITE ? seg_off[l] : 0;
    int nseg = 0;
    walk_segments<BIN>(L, l, g, flags, [&](const Segment<T> &cur, int tl) {
        const int sid = base + nseg;
        if (WRITE) segs[sid] = cur;
        if (BIN) {
            for (int tb = cur.lo >> g.tile_log; tb <= cur.hi >> g.tile_log; tb++) {
                const int64_t tid = tile_index(g, L.frame, L.axis, tl, tb);
                if (!WRITE) atomicAdd(&tile_cnt[tid], 1);
                else items[tile_off[tid] + atomicAdd(&tile_cur[tid], 1)] = sid;
            }
        }
        nseg++;
    });
    if (!WRITE) seg_cnt[l] = nseg;
}

// Unordered plan (the tile path, whose result does not depend on segment
// order): one walk per line.
//   k_setup_lines   line constants, flags, and the total of the per-line
//                   segment bounds (counters[0]);
//   k_walk_lines    orders the workgroup's lines by segment bound, takes
//                   slots for their bounds with one atomic (counters[1]),
//                   walks, writes the segments into them (unused slots get
//                   ncols = 0) and counts tile items (atomics the walk does
//                   not wait for);
//   k_bin_slots     one lane per slot: writes the per-tile item lists, one
//                   cursor atomic per run of a tile's slots in a wave.
template <typename T, typename I>
__global__ void __launch_bounds__(256)
k_setup_lines(const T *__restrict__ lines, const I *__restrict__ idxs, const uint8_t *__restrict__ kernels,
              int kernel, int64_t n_lines, Geometry g, LineSetup<T> *__restrict__ setup,
              LineLite *__restrict__ lite, unsigned long long *__restrict__ counters, int *__restrict__ flags)
{
    const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int ub = 0;
    if (l < n_lines) {
        LineSetup<T> L;
        setup_line(lines, idxs, kernels, kernel, l, g, L, flags);
        setup[l] = L;
        if constexpr (sizeof(T) == 4) lite[l] = line_lite(L);
        ub = segment_bound(L, g);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ub += __shfl_xor(ub, o, 64);
    // one global atomic per workgroup (same-address atomics serialise)
    __shared__ unsigned long long bsum;
    if (threadIdx.x == 0) bsum = 0ull;
    __syncthreads();
    if ((threadIdx.x & 63) == 0 && ub) atomicAdd(&bsum, (unsigned long long)ub);
    __syncthreads();
    if (threadIdx.x == 0 && bsum) atomicAdd(&counters[0], bsum);
}

template <typename T>
__global__ void __launch_bounds__(256)
k_walk_lines(int64_t n_lines, Geometry g, const LineSetup<T> *__restrict__ setup, Segment<T> *__restrict__ segs,
             int64_t slot_cap, unsigned long long *__restrict__ counters, int *__restrict__ tile_cnt,
             int *__restrict__ flags, int64_t *__restrict__ line_base)
{
    const int64_t l0 = (int64_t)blockIdx.x * blockDim.x;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6, n_waves = (blockDim.x + 63) >> 6;
    LineSetup<T> L;
    int ub = 0;
    int64_t l = l0 + threadIdx.x;
    if (l < n_lines) {
        L = setup[l];
        ub = segment_bound(L, g);
    }
    {
        // A wave steps until its longest walk ends.  The workgroup's lines
        // are ordered by segment bound (min(bound, 63); a stable LSD radix
        // sort of one bit per pass, ballot splits), so that each wave walks
        // lines of similar length; thread t then walks the t-th line.
        __shared__ int s_ub[256], s_id[256], s_zero[4];
        int id = threadIdx.x;
        const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
        for (int bit = 0; bit < 6; bit++) {
            const bool one = (min(ub, 63) >> bit) & 1;
            const uint64_t zm = __ballot(!one);
            const int zb = __popcll(zm & below);
            if (lane == 0) s_zero[wave] = __popcll(zm);
            __syncthreads();
            int zt = 0, zw = 0;
            for (int w = 0; w < n_waves; w++) {
                const int z = s_zero[w];
                zw += (w < wave) ? z : 0;
                zt += z;
            }
            // zeros keep their order in front, ones after them
            const int pos = one ? zt + (wave * 64 - zw) + (lane - zb) : zw + zb;
            s_ub[pos] = ub;
            s_id[pos] = id;
            __syncthreads();
            ub = s_ub[threadIdx.x];
            id = s_id[threadIdx.x];
        }
        l = l0 + id;
        if (ub > 0) L = setup[l];
    }
    // wave prefix of the bounds, one slot reservation per wave
    int pre = ub;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(pre, d, 64);
        if (lane >= d) pre += y;
    }
    const int total = __shfl(pre, 63, 64);
    pre -= ub;
    // slots for the workgroup's waves with one global atomic (same-address
    // atomics serialise), handed out in wave order
    __shared__ unsigned long long wsum[4];
    if (lane == 0) wsum[wave] = (unsigned long long)total;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long bt = 0;
        for (int w = 0; w < n_waves; w++) bt += wsum[w];
        unsigned long long b = bt ? atomicAdd(&counters[1], bt) : 0ull;
        if (bt && (int64_t)(b + bt) > slot_cap) atomicOr(flags, FLAG_OVERFLOW);
        for (int w = 0; w < n_waves; w++) {
            const unsigned long long t = wsum[w];
            wsum[w] = b;
            b += t;
        }
    }
    __syncthreads();
    const unsigned long long wbase = wsum[wave];
    // first slot of each line (the adjoint's per-line reduction)
    if (line_base && l < n_lines) line_base[l] = (int64_t)wbase + pre;
    if (ub == 0 || (int64_t)(wbase + total) > slot_cap) return;
    const int64_t base = (int64_t)wbase + pre;
    int nseg = 0;
    // The tile counts are atomics whose results the walk does not use
    // (k_bin_slots places the items); each lane adds up runs of items into
    // the same list (consecutive segments of a line mostly share their tiles)
    // in two pending counters and issues one atomic per run.
    int pend_a = -1, pend_b = -1, n_a = 0, n_b = 0;   // pending list counts (list index, items)
    Segment<T> *const dst = segs + base;
    // (axis 0: the long axis runs along tile columns)
    const int fbase = L.frame * (g.nty * g.ntx), ml = (L.axis == 0) ? 1 : g.ntx, mb = (L.axis == 0) ? g.ntx : 1;
    walk_segments<false>(L, l, g, flags, [&](const Segment<T> &cur, int tl) {
        if (nseg < ub) dst[nseg] = cur;
        const int tb0 = cur.lo >> g.tile_log, tb1 = cur.hi >> g.tile_log;
        int li = (fbase + tl * ml + tb0 * mb) * LIST_SUBS + L.sub;
        for (int tb = tb0; tb <= tb1; tb++, li += mb * LIST_SUBS) {
            if (li == pend_a) {
                n_a++;
            } else if (li == pend_b) {
                n_b++;
            } else {
                if (n_b) atomicAdd(&tile_cnt[pend_b], n_b);
                pend_b = pend_a;
                n_b = n_a;
                pend_a = li;
                n_a = 1;
            }
        }
        nseg++;
    });
    if (n_a) atomicAdd(&tile_cnt[pend_a], n_a);
    if (n_b) atomicAdd(&tile_cnt[pend_b], n_b);
    if (nseg > ub) atomicOr(flags, FLAG_STUCK); // cannot happen: the bound holds for every walk
    for (int k = nseg; k < ub; k++) segs[base + k].ncols = 0;
}

// Clears a plan's counters before a draw (a kernel, not a memset: a draw may
// be captured in a HIP graph).
__global__ void k_plan_reset(int64_t n_lists, unsigned long long *__restrict__ counters, int *__restrict__ flags,
                             int *__restrict__ cnt, int *__restrict__ cur, unsigned long long *__restrict__ scan_state,
                             int64_t scan_words)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < scan_words) scan_state[i] = 0ull;
    if (i == 0) {
        counters[0] = 0ull;
        counters[1] = 0ull;
        *flags = 0;
    }
    if (i < n_lists) {
        cnt[i] = 0;
        cur[i] = 0;
    }
}

// The list of a tile's sub-list: a run of lanes (consecutive slots) whose segments
// reach it takes its places with one cursor atomic, in lane order, so a list
// holds runs of consecutive slots (the tile kernels' segment loads coalesce).
// Neighbours are all that needs comparing: consecutive segments of a line mostly
// share their tiles, different lines seldom do.
//
// Bound by the atomics (about 20 G requests/s): 300 us for 962 000 lines, 318
// with a loop over the distinct tiles of the wave; two and four groups of slots
// per lane, with their loads in flight together, took 312 and 338.
template <typename T>
__global__ void __launch_bounds__(256)
k_bin_slots(int64_t n_slots, Geometry g, const LineSetup<T> *__restrict__ setup, const Segment<T> *__restrict__ segs,
            const int *__restrict__ tile_off, int *__restrict__ cur, int2 *__restrict__ pairs,
            const unsigned long long *__restrict__ counters, int64_t n_tiles, int64_t item_cap,
            int *__restrict__ flags, int *__restrict__ slot_tiles)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    // after a slot overflow some reserved slots were never written (stale
    // segments): bin nothing; otherwise the slots taken by the walk, and the
    // item total against the list capacity
    const int fl = *flags, items = tile_off[n_tiles * LIST_SUBS];
    const int64_t taken = min(n_slots, (int64_t)counters[1]);
    if (fl & FLAG_OVERFLOW) return;
    if ((int64_t)items > item_cap) {
        if (i == 0) atomicOr(flags, FLAG_OVERFLOW);
        return;
    }
    int np = 0, li = 0, step = 0;   // tiles of the slot, list index of the first, distance to the next
    int2 item = make_int2(0, 0);
    if (i < taken) {
        const Segment<T> sg = segs[i];
        if (sg.ncols > 0) {
            const LineSetup<T> &L = setup[sg.line];
            const int axis = L.axis, frame = L.frame, sub = L.sub;
            const int tl = pick(sg.c, axis) >> g.tile_log, tb = sg.lo >> g.tile_log;
            np = (sg.hi >> g.tile_log) - tb + 1;
            li = (int)tile_index(g, frame, axis, tl, tb) * LIST_SUBS + sub;
            step = ((axis == 0) ? g.ntx : 1) * LIST_SUBS;
            item = make_int2((int)i, sg.line);
        }
    }
    // tiles per slot, for the adjoint's partial sums (0 for unused slots)
    if (slot_tiles && i < n_slots) slot_tiles[i] = np;
    // two tiles of each slot per turn
    for (int p = 0; __ballot(p < np) != 0ull; p += 2) {
        int key[2], head[2], off[2], b[2];
#pragma unroll
        for (int v = 0; v < 2; v++) {
            key[v] = (p + v < np) ? li + (p + v) * step : -1;
            off[v] = (key[v] >= 0) ? tile_off[key[v]] : 0;
            const int left = __shfl_up(key[v], 1, 64);   // (every lane of the wave takes part)
            const uint64_t heads = __ballot((lane == 0) | (key[v] != left));
            const uint64_t upto = ~0ull >> (63 - lane), rest = heads & ~upto;
            head[v] = 63 - __builtin_clzll(heads & upto);
            b[v] = 0;
            if ((key[v] >= 0) & (lane == head[v]))
                b[v] = atomicAdd(&cur[key[v]], (rest ? __builtin_ctzll(rest) : 64) - lane);
        }
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const int at = off[v] + __shfl(b[v], head[v], 64) + lane - head[v];
            if (key[v] >= 0) pairs[at] = item;
        }
    }
}

// ---------------------------------------------------------------------------
// emission pass (pixel lists and the deterministic mode)
// ---------------------------------------------------------------------------
template <typename T, int K, bool WRITE>
__global__ void __launch_bounds__(256)
k_emit(const Segment<T> *__restrict__ segs, int64_t n_segs, const LineSetup<T> *__restrict__ setup, int H, int W,
       T max_val, int *__restrict__ cnt, const int64_t *__restrict__ off, uint64_t *__restrict__ keys,
       T *__restrict__ vals, int32_t *__restrict__ lines_out, int *__restrict__ flags)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_segs) return;
    const Segment<T> sg = segs[i];
    const LineSetup<T> L = setup[sg.line];
    const int a = L.axis, b = 1 - a, sa = pick(L.st, a);
    const int db = (b == 0) ? W : H;
    const int64_t base = WRITE ? off[i] : 0;
    int n = 0;

    WalkState<T> s;
    s.c[0] = sg.c[0];
    s.c[1] = sg.c[1];
    s.Te = sg.Te;
    s.Ne = sg.Ne;
    const int c0 = pick(s.c, a);
    int it = 0;
    for (; it < 4 * 64 + 16; it++) {
        if (walk_done(L, s)) break;
        const int k = (pick(s.c, a) - c0) * sa;
        if (k >= sg.ncols) break;
        bool nx, ny;
        walk_next(L, s.Ne, nx, ny);
        if ((a == 0) ? nx : ny) {
            ColRec<T> cr;
            cr.s = pick(s.c, b);
            cr.Te = s.Te;
            cr.Ne = s.Ne;
            const int c = pick(s.c, a);
            fill_column(L, cr, 0, db, [&](int sp, T Te, T Ne) {
                const T err = err_of(L, Te, Ne);
                if (!(err <= T(1))) return;
                if (WRITE) {
                    const int x = (a == 0) ? c : sp, y = (a == 0) ? sp : c;
                    keys[base + n] = ((uint64_t)L.frame * (uint64_t)H + (uint64_t)y) * (uint64_t)W + (uint64_t)x;
                    vals[base + n] = pixel_value<K>(err, max_val);
                    if (lines_out) lines_out[base + n] = sg.line;
                }
                n++;
            });
        }
        walk_step(L, s, nx, ny);
    }
    if (it == 4 * 64 + 16) atomicOr(flags, FLAG_STUCK);
    if (!WRITE) cnt[i] = n;
}

__global__ void k_i32_to_i64(const int *__restrict__ in, int64_t *__restrict__ out, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[i];
}

template <typename T>
__global__ void k_raw_out(const uint64_t *__restrict__ keys, const T *__restrict__ vals,
                          const int32_t *__restrict__ line_of, int64_t n, int64_t H, int64_t W,
                          int32_t *__restrict__ of, int32_t *__restrict__ oy, int32_t *__restrict__ ox,
                          T *__restrict__ ov, int32_t *__restrict__ ol)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t key = keys[i];
    const uint64_t hw = (uint64_t)H * (uint64_t)W;
    of[i] = (int32_t)(key / hw);
    const uint64_t r = key % hw;
    oy[i] = (int32_t)(r / (uint64_t)W);
    ox[i] = (int32_t)(r % (uint64_t)W);
    ov[i] = vals[i];
    if (ol) ol[i] = line_of[i];
}

// ---------------------------------------------------------------------------
// ordered (reference-order) accumulation: deterministic images and merged
// pixel lists
// ---------------------------------------------------------------------------

// Sorts each tile's item list by segment id, i.e. by (line, walk position):
// the order in which the reference's single thread visits the segments.
// One workgroup per tile, bitonic sort in LDS.
constexpr int SORT_MAX = 8192;
constexpr int FLAG_TILE_FULL = 8;

__global__ void __launch_bounds__(256)
k_sort_tile_items(const int *__restrict__ tile_off, int *__restrict__ items, int *__restrict__ flags,
                  const int *__restrict__ tile_list)
{
    __shared__ int buf[SORT_MAX];
    const int tile = tile_list ? tile_list[blockIdx.x] : (int)blockIdx.x;
    const int beg = tile_off[tile], n = tile_off[tile + 1] - beg;
    if (n <= 1) return;
    if (n > SORT_MAX) {
        if (threadIdx.x == 0) atomicOr(flags, FLAG_TILE_FULL);
        return;
    }
    int p2 = 2;
    while (p2 < n) p2 <<= 1;
    for (int i = threadIdx.x; i < p2; i += blockDim.x) buf[i] = (i < n) ? items[beg + i] : INT_MAX;
    __syncthreads();
    for (int k = 2; k <= p2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < p2; i += blockDim.x) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const int a = buf[i], b = buf[ixj];
                    const bool up = (i & k) == 0;
                    if ((a > b) == up) {
                        buf[i] = b;
                        buf[ixj] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) items[beg + i] = buf[i];
}

// One wave per tile.  Items are applied one at a time in sorted order; the
// lanes of an item cover its columns (no pixel repeats inside one line), so
// every pixel sees its contributions in ascending line order, starting from
// the value already in the frame (image mode) or from its first contribution
// (list mode: `first` records the first contributing line).
__device__ inline unsigned int val_bits(float v) { return __float_as_uint(v); }
__device__ inline unsigned long long val_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
__device__ inline float bits_val(unsigned int b, float) { return __uint_as_float(b); }
__device__ inline double bits_val(unsigned long long b, double) { return __longlong_as_double((long long)b); }

// *p = max(*p, v) in the order std::max(*p, v) takes: replaced only if *p < v
__device__ inline void atomic_max_val(float *p, float v)
{
    unsigned int *q = (unsigned int *)p;
    unsigned int old = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (bits_val(old, v) < v) {
        const unsigned int prev = atomicCAS(q, old, val_bits(v));
        if (prev == old) break;
        old = prev;
    }
}

__device__ inline void atomic_max_val(double *p, double v)
{
    unsigned long long *q = (unsigned long long *)p;
    unsigned long long old = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (bits_val(old, v) < v) {
        const unsigned long long prev = atomicCAS(q, old, val_bits(v));
        if (prev == old) break;
        old = prev;
    }
}

// ACC >= 0 (accumulate_lines): the plan's frames are terms; every touched
// pixel of a term tile (accumulated from zero, as with LIST) is combined into
// frame term_frame[term] of img with atomics, sum (ACC 0) or max (ACC 1).
template <typename T, int K, int OV, int TILE, int SEG, bool LIST, int ACC>
__global__ void __launch_bounds__(64)
k_tiles_ordered(T *__restrict__ img, uint8_t *__restrict__ touched, int32_t *__restrict__ first_line, Geometry g,
                const int *__restrict__ tile_off, const int *__restrict__ items, const Segment<T> *__restrict__ segs,
                const LineSetup<T> *__restrict__ setup, T max_val, int *__restrict__ flags,
                const int32_t *__restrict__ term_frame, const int *__restrict__ tile_list)
{
    static_assert(ACC < 0 || LIST, "accumulation starts from zero");
    static_assert(2 * SEG <= 64, "two lanes per column");
    __shared__ T acc[TILE * TILE];
    __shared__ int32_t first[TILE * TILE];
    __shared__ ColRec<T> rec[64 * SEG];
    __shared__ ItemHdr hdr[64];

    const int tile = tile_list ? tile_list[blockIdx.x] : (int)blockIdx.x;
    const int beg = tile_off[tile], end = tile_off[tile + 1];
    // a tile too large to sort (k_sort_tile_items, earlier on the stream)
    // fails the call: leave every output untouched
    if (beg == end || (__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_TILE_FULL))
        return;
    const int per_frame = g.ntx * g.nty;
    const int64_t f = tile / per_frame;
    const int r = tile - (int)f * per_frame;
    const int ty = r / g.ntx, tx = r - ty * g.ntx;
    const int X0 = tx * TILE, Y0 = ty * TILE;
    const int X1 = min(X0 + TILE, g.W), Y1 = min(Y0 + TILE, g.H);
    T *fo = ACC >= 0 ? img : img + (f * g.H) * (int64_t)g.W;
    const int lane = threadIdx.x;

    for (int i = lane; i < TILE * TILE; i += 64) {
        const int y = Y0 + i / TILE, x = X0 + (i % TILE);
        if (LIST) acc[i] = T(0);
        else acc[i] = (y < Y1 && x < X1) ? fo[(int64_t)y * g.W + x] : T(0);
        first[i] = -1;
    }
    wave_sync();

    for (int c0 = beg; c0 < end; c0 += 64) {
        const int n = min(64, end - c0);
        if (lane < n) {
            const int sid = items[c0 + lane];
            const Segment<T> sg = segs[sid];
            const LineSetup<T> L = setup[sg.line];
            hdr[lane].seg = sid;
            hdr[lane].line = sg.line;
            walk_columns<T, SEG>(L, sg, rec, lane, flags);
        }
        wave_sync();
        for (int j = 0; j < n; j++) {
            if (lane < 2 * SEG) {
                const int k = lane >> 1, half = lane & 1;
                const ColRec<T> cr = rec[j * SEG + k];
                if (cr.s != INT_MIN) {
                    const Segment<T> &sg = segs[hdr[j].seg];
                    const LineSetup<T> &L = setup[hdr[j].line];
                    const int line = hdr[j].line;
                    const int a = L.axis, b = 1 - a;
                    const int c = pick(sg.c, a) + k * pick(L.st, a);
                    const int s_lo = (a == 0) ? Y0 : X0, s_hi = (a == 0) ? Y1 : X1;
                    auto put = [&](int s, T Te, T Ne) {
                        const T err = err_of(L, Te, Ne);
                        if (!(err <= T(1))) return;
                        const int x = (a == 0) ? c : s, y = (a == 0) ? s : c;
                        const int p = (y - Y0) * TILE + (x - X0);
                        const T v = pixel_value<K>(err, max_val);
                        if (LIST && first[p] < 0) {
                            first[p] = line;
                            // accumulate_lines' term buffer starts at zero: 0 + v, or
                            // std::max(0, v) (bresenham.cpp:218-221)
                            acc[p] = (ACC < 0) ? v : ((OV == 0) ? T(0) + v : ((T(0) < v) ? v : T(0)));
                        } else {
                            if (OV == 0) acc[p] = acc[p] + v;
                            else acc[p] = (acc[p] < v) ? v : acc[p];
                            if (!LIST && first[p] < 0) first[p] = line;
                        }
                    };
                    // lane pair (k, 0): centre and the +step half; (k, 1): the -step half
                    if (half == 0 && cr.s >= s_lo && cr.s < s_hi) put(cr.s, cr.Te, cr.Ne);
                    const int dir = half ? -pick(L.st, b) : pick(L.st, b);
                    const T dT = (dir > 0) ? pick(L.t, b) : -pick(L.t, b), dN = (dir > 0) ? pick(L.nv, b) : -pick(L.nv, b);
                    int s = cr.s;
                    T Te = cr.Te, Ne = cr.Ne;
                    for (;;) {
                        s += dir;
                        Te += dT;
                        Ne += dN;
                        if (!(nsq_of(L, Ne) < L.w2)) break;
                        if (s >= s_lo && s < s_hi) put(s, Te, Ne);
                        else if ((dir > 0) ? (s >= s_hi) : (s < s_lo)) break;
                    }
                }
            }
            wave_sync();
        }
    }

    for (int i = lane; i < TILE * TILE; i += 64) {
        const int y = Y0 + i / TILE, x = X0 + (i % TILE);
        if (y >= Y1 || x >= X1) continue;
        const int64_t o = (int64_t)y * g.W + x;
        if (ACC >= 0) {
            if (first[i] >= 0) {
                T *dst = img + ((int64_t)term_frame[f] * g.H) * (int64_t)g.W + o;
                if (ACC == 0) atomicAdd(dst, acc[i]);
                else atomic_max_val(dst, acc[i]);
            }
        } else if (LIST) {
            const int64_t q = (f * g.H) * (int64_t)g.W + o;
            touched[q] = first[i] >= 0;
            if (first[i] >= 0) {
                fo[o] = acc[i];
                if (first_line) first_line[q] = first[i];
            }
        } else if (first[i] >= 0) {
            fo[o] = acc[i];
        }
    }
}

// stream compaction of a dense (image, touched) pair in raster order
__global__ void k_row_count(const uint8_t *__restrict__ touched, int64_t rows, int W, int64_t *__restrict__ cnt)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const uint8_t *t = touched + r * W;
    int64_t c = 0;
    for (int x = 0; x < W; x++) c += t[x];
    cnt[r] = c;
}

template <typename T>
__global__ void k_row_write(const uint8_t *__restrict__ touched, const T *__restrict__ img,
                            const int32_t *__restrict__ first_line, int64_t rows, int H, int W,
                            const int64_t *__restrict__ off, int32_t *__restrict__ of, int32_t *__restrict__ oy,
                            int32_t *__restrict__ ox, T *__restrict__ ov, int32_t *__restrict__ ol)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    int64_t p = off[r];
    const int64_t base = r * W;
    for (int x = 0; x < W; x++) {
        if (!touched[base + x]) continue;
        of[p] = (int32_t)(r / H);
        oy[p] = (int32_t)(r % H);
        ox[p] = x;
        ov[p] = img[base + x];
        if (ol) ol[p] = first_line[base + x];
        p++;
    }
}

// ---------------------------------------------------------------------------
// adjoint (sum overlap): per (segment, tile) partial gradients, then an
// ordered per-line reduction
// ---------------------------------------------------------------------------
// Per-line constants of the per-pixel gradient terms (double).  The tangent
// is the exact difference of the end points (the walk's float tangent
// p1 - p0 is rounded, which moves dist by ~1e-5 relative at these
// magnitudes); cc and cw fold max_val, the profile's constant and the powers
// of 1/w of the two gradient factors (see pixel_grad).
struct GradConst {
    double x0, y0, tx, ty, inv_mag, inv_w2, cc, cw;
};

template <int K, typename T>
__device__ __forceinline__ GradConst grad_const(const LineSetup<T> &L, const T *line, T max_val)
{
    GradConst c;
    c.x0 = (double)L.p0[0];
    c.y0 = (double)L.p0[1];
    c.tx = (double)line[2] - c.x0;
    c.ty = (double)line[3] - c.y0;
    c.inv_mag = 1.0 / (c.tx * c.tx + c.ty * c.ty);
    const double inv_w = 1.0 / (double)L.w;
    c.inv_w2 = inv_w * inv_w;
    const double mv = (double)max_val;
    // K(sqrt(u)) = k(u): dK/d(dist^2) = k'(u) / w^2 and dK/dw = k'(u) (-2 u / w);
    // k'(u) = -1.875 (1 - u) (biweight), -0.75 (parabolic), -4.5 k(u) (gaussian)
    double kp;
    if constexpr (K == K_BIWEIGHT) kp = -1.875;
    else if constexpr (K == K_PARABOLIC) kp = -0.75;
    else if constexpr (K == K_GAUSSIAN) kp = -4.5 * 0.3989422804014327;
    else kp = 0.0;
    if constexpr (K == K_TRIANGULAR) {
        // K = 1 - dist / w: dK/d(dist^2) = -1 / (2 w dist), dK/dw = dist / w^2
        c.cc = mv * inv_w;
        c.cw = mv * c.inv_w2;
    } else {
        c.cc = -2.0 * kp * mv * c.inv_w2;
        c.cw = -2.0 * kp * mv * inv_w;
    }
    return c;
}

// Per-pixel gradient terms of max_val K(dist / w), in double.  With q the
// clamped projection of p (parameter ts in [0, 1]) and (dx, dy) = p - q,
// d(dist^2)/d(x0, y0) = -2 (1 - ts) (dx, dy) and d(dist^2)/d(x1, y1) =
// -2 ts (dx, dy).  The accumulators hold
//   acc[0..1] = sum c (dx, dy),  acc[2..3] = sum c ts (dx, dy),  acc[4] = dL/dw,
// with c = -2 g max_val dK/d(dist^2); the end-point gradients are then
// (acc[0] - acc[2], acc[1] - acc[3], acc[2], acc[3]) (grad_finish).
template <int K>
__device__ __forceinline__ void pixel_grad(const GradConst &C, int x, int y, double gv, double *acc)
{
    const double rx = (double)x - C.x0, ry = (double)y - C.y0;
    double ts = __builtin_fma(ry, C.ty, rx * C.tx) * C.inv_mag;
    ts = (ts < 0.0) ? 0.0 : ((ts > 1.0) ? 1.0 : ts);
    const double dx = __builtin_fma(-ts, C.tx, rx), dy = __builtin_fma(-ts, C.ty, ry);
    const double d2 = __builtin_fma(dx, dx, dy * dy);
    double c, gw;
    if constexpr (K == K_TRIANGULAR) {
        const double dist = sqrt(d2);
        c = (dist > 0.0) ? gv * C.cc / dist : 0.0;
        gw = gv * dist;
    } else {
        const double u = d2 * C.inv_w2;
        double f;   // k'(u) / k'(0)
        if constexpr (K == K_BIWEIGHT) f = 1.0 - u;
        else if constexpr (K == K_GAUSSIAN) f = ::exp(-4.5 * u);
        else f = 1.0;
        const double gf = gv * f;
        c = gf * C.cc;
        gw = gf * u;
    }
    const double cts = c * ts;
    acc[0] = __builtin_fma(c, dx, acc[0]);
    acc[1] = __builtin_fma(c, dy, acc[1]);
    acc[2] = __builtin_fma(cts, dx, acc[2]);
    acc[3] = __builtin_fma(cts, dy, acc[3]);
    acc[4] = __builtin_fma(gw, C.cw, acc[4]);
}

// LDS row pitch of the adjoint's gradient tile, in words: 4 words of padding
// per row.  The lanes of one item read the same short-axis coordinate in 8 or
// 16 consecutive rows (steep lines); with a pitch of TILE (a multiple of the
// bank count) those reads fall in one bank, with TILE + 4 in distinct banks.
// (k_tiles_fast pads its rows alike; k_tiles does not, where padding spilled.)
template <int TILE>
constexpr int tile_pitch() { return TILE + 4; }

// The sums of one column's gradient terms.  With (a, b) the line's long and
// short axes, r = p - p0, t the exact tangent, q = r_a t_b - r_b t_a and T = r t
// (both linear along the column), Tc = T clamped to [0, |t|^2] and o = T - Tc, a
// pixel's vector from its projection is (q (t_b, -t_a) + o (t_a, t_b)) / |t|^2,
// its dist^2 is (q^2 + o^2) / |t|^2 and its ts is Tc / |t|^2.  The terms of
// pixel_grad are constants of the line times these sums:
//   s[0] = sum h q,  s[1] = sum h q Tc,  s[2] = sum g k,
//   s[3] = sum h o,  s[4] = sum h o Tc   (zero for columns within the ends)
// with h = g f, k = f u (u = dist^2 / w^2, ku = 1 / (|t| w)^2); triangular
// profiles: h = g / r, k = r = sqrt(q^2 + o^2).
template <int K>
__device__ __forceinline__ void add_inside(double *s, float g, double q, double T, double ku)
{
    const double gv = (double)g;
    if constexpr (K == K_TRIANGULAR) {
        const double p = (q > 0.0) ? gv : ((q < 0.0) ? -gv : 0.0);
        s[0] += p;
        s[1] = __builtin_fma(p, T, s[1]);
        s[2] = __builtin_fma(gv, __builtin_fabs(q), s[2]);
    } else {
        const double u = q * q * ku;
        double h = gv;
        if constexpr (K == K_BIWEIGHT) h = __builtin_fma(-u, gv, gv);
        if constexpr (K == K_GAUSSIAN) h = gv * ::exp(-4.5 * u);
        const double p = h * q;
        s[0] += p;
        s[1] = __builtin_fma(p, T, s[1]);
        s[2] = __builtin_fma(h, u, s[2]);
    }
}

template <int K>
__device__ __forceinline__ void add_clamped(double *s, float g, double q, double T, double mag, double ku)
{
    const double gv = (double)g;
    const double Tc = (T < 0.0) ? 0.0 : ((T > mag) ? mag : T), o = T - Tc;
    const double r2 = __builtin_fma(q, q, o * o);
    double h = gv, k;
    if constexpr (K == K_TRIANGULAR) {
        k = sqrt(r2);
        h = (k > 0.0) ? gv / k : 0.0;
        s[2] = __builtin_fma(gv, k, s[2]);
    } else {
        k = r2 * ku;
        if constexpr (K == K_BIWEIGHT) h = __builtin_fma(-k, gv, gv);
        if constexpr (K == K_GAUSSIAN) h = gv * ::exp(-4.5 * k);
        s[2] = __builtin_fma(h, k, s[2]);
    }
    const double p = h * q, e = h * o;
    s[0] += p;
    s[1] = __builtin_fma(p, Tc, s[1]);
    s[3] += e;
    s[4] = __builtin_fma(e, Tc, s[4]);
}

// x of the lane at a fixed place of the row of 16 (CTRL: a DPP control), and the
// sum of x over the SEG lanes of an item, in the same order in every lane
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int SEG>
__device__ __forceinline__ double item_sum(double x)
{
    static_assert(SEG == 8 || SEG == 16, "lanes of one row");
    x += dpp_move<0xb1>(x);    // lanes 1, 0, 3, 2
    x += dpp_move<0x4e>(x);    // lanes 2, 3, 0, 1
    x += dpp_move<0x141>(x);   // mirrored within 8
    if constexpr (SEG == 16) x += dpp_move<0x140>(x);   // mirrored within 16
    return x;
}

// Per-item record of k_adjoint_fast in LDS.
struct AdjRec {
    double q0, T0;      // q and T at column 0 and short-axis coordinate 0
    double la, lb;      // t_a, t_b (exact: from the end points)
    double ku;          // 1 / (|t| w)^2
    float inv;          // 1 / nb: nb is the normal error's change per +1 along the short axis
    float hm, hp;       // half height of the band in steps: decided inside, decided outside
    float cap, far;     // interior columns: cap < Te < far
    int32_t base;       // LDS index of column 0 at short-axis coordinate 0
    int32_t s0;         // short-axis position at column 0
    int32_t line;
    int32_t meta;       // FR_* bits, columns from bit 16
};

// Adjoint of the float lines.  One workgroup per tile, NT / 64 independent
// waves (the only barrier is after the tile of dLoss/dImage is in LDS), each
// with chunks of up to CHW items: phase 1 replays one item's walk per lane;
// phase 2a gives a lane one interior column, its pixels counted beforehand as
// in the tile kernel of the draws and its terms reduced to three sums;
// phase 2b takes the columns within the width of a line's end from a compacted
// list, one half per lane, with the error of every pixel and the terms of
// pixels beyond the end.  Lane i collects item i: the columns of phase 2a in a
// fixed tree, those of phase 2b in their order, so a partial does not depend on
// where its item stands in the list.
//
// Bound by vector instruction issue: the gradient of 160 000 biweight lines
// (widths 2 to 6, 32 frames of 1024^2) takes 584 us, of which its 289 M wave
// instructions need 470 at the issue rate; with one lane per column and the
// full terms (25 double operations, two divisions per column) 983 us.  Chunks of
// 16 items leave half the lanes of phase 2b idle (838 against 688 us with 32,
// before the sums of phase 2b were shared with 2a); 192 / SEG fill four
// workgroups of 40 KB per CU.
template <int K, int TILE, int SEG, int NT, int CHW>
__global__ void __launch_bounds__(NT, 4)
k_adjoint_fast(const float *__restrict__ grad, const float *__restrict__ lines, Geometry g,
               const int *__restrict__ tile_off, const int2 *__restrict__ pairs,
               const Segment<float> *__restrict__ segs, const LineSetup<float> *__restrict__ setup,
               const LineLite *__restrict__ lite, const int *__restrict__ slot_base, float max_val,
               double *__restrict__ partial, int *__restrict__ flags)
{
    constexpr int NW = NT / 64, PX = TILE * TILE, PITCH = tile_pitch<TILE>(), NREC = CHW * SEG;
    constexpr int IPR = 64 / SEG;   // items per round of phase 2a
    constexpr int BATCH = 32;       // columns per round of phase 2b
    static_assert(CHW <= 64 && NREC <= 256, "one lane per item, column numbers of 8 bits");
    union Sums {   // per wave: the items' sums of phase 2a, then the columns' of phase 2b
        double item[CHW][3];
        double col[BATCH][5];
    };
    __shared__ float gt[TILE * PITCH];
    __shared__ WaveCols<NREC> cols[NW];
    __shared__ AdjRec arec[NW][CHW];
    __shared__ uint8_t caps[NW][NREC];
    __shared__ Sums sums[NW];

    const int tile = blockIdx.x;
    const int beg = tile_off[tile * LIST_SUBS], end = tile_off[(tile + 1) * LIST_SUBS];
    // a plan whose last draw failed (capacity, bad idxs) has no valid lists
    const int fl = *flags;
    if (fl || beg == end) return;
    int64_t f;
    int tx, ty;
    tile_coords(g, tile, f, tx, ty);
    const int X0 = tx * TILE, Y0 = ty * TILE;
    const int X1 = min(X0 + TILE, g.W), Y1 = min(Y0 + TILE, g.H);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // the tile of dLoss/dImage: every load issued before the LDS writes
    const float *const fg = grad + ((f * g.H + Y0) * (int64_t)g.W + X0);
    constexpr int PP = PX / NT;
    float gv[PP];
    // (rows below the frame, which no fill reaches, are left out four of the wave's at a time)
    auto inside = [&](int j) { return (wave * 64 + j * NT) / TILE < Y1 - Y0; };
    static_assert(PP % 4 == 0, "groups of 4");
#pragma unroll
    for (int j0 = 0; j0 < PP; j0 += 4) {
        if (!inside(j0)) continue;
#pragma unroll
        for (int j = j0; j < j0 + 4; j++) {
            const int i = tid + j * NT;
            const int y = i / TILE, x = i % TILE;
            gv[j] = (y < Y1 - Y0 && x < X1 - X0) ? __builtin_nontemporal_load(fg + ((int64_t)y * g.W + x)) : 0.0f;
        }
    }
    // equal chunks, the same number of turns for every wave
    const int turns = (end - beg + NW * CHW - 1) / (NW * CHW);
    const int size = (end - beg + turns * NW - 1) / (turns * NW);
    Segment<float> sg;
    LineLite L;
    float ln[5];
    int sbase;
    auto take = [&](const int2 &it) {
        sg = segs[it.x];
        L = lite[it.y];
        sbase = slot_base[it.x];
        for (int k = 0; k < 5; k++) ln[k] = lines[5 * (int64_t)it.y + k];
    };
    // (lanes without an item load the list's last)
    take(pairs[min(beg + wave * size + lane, end - 1)]);
#pragma unroll
    for (int j0 = 0; j0 < PP; j0 += 4) {
        if (!inside(j0)) continue;
#pragma unroll
        for (int j = j0; j < j0 + 4; j++) {
            const int i = tid + j * NT;
            gt[(i / TILE) * PITCH + (i % TILE)] = gv[j];
        }
    }
    __syncthreads();

    WaveCols<NREC> &wK = cols[wave];
    AdjRec *const wR = arec[wave];
    uint8_t *const wC = caps[wave];
    Sums &wX = sums[wave];
    const uint64_t below = (1ull << lane) - 1ull;

    for (int t = 0; t < turns; t++) {
        const int first = beg + (t * NW + wave) * size;
        const int n = min(size, end - first);
        if (n <= 0) break;
        const int2 np = pairs[min(first + NW * size + lane, end - 1)];   // the next turn's items
        // phase 1 (as in k_tiles_fast)
        const bool ax = L.meta & FR_AXIS;
        const double la = (double)ln[ax ? 3 : 2] - (double)ln[ax ? 1 : 0];
        const double lb = (double)ln[ax ? 2 : 3] - (double)ln[ax ? 0 : 1];
        const double inv_mag = 1.0 / (la * la + lb * lb), inv_w = 1.0 / (double)ln[4];
        const int64_t out_at = (int64_t)sbase + ((ax ? tx : ty) - (sg.lo >> g.tile_log));
        if (lane < n) {
            const float nb = ax ? L.t[1] : -L.t[0], na = __builtin_fabsf(nb);
            const int c0 = ax ? sg.c[1] : sg.c[0];
            const double ra = (double)c0 - (double)ln[ax ? 1 : 0], rb = -(double)ln[ax ? 0 : 1];
            AdjRec R;
            R.q0 = ra * lb - rb * la;
            R.T0 = ra * la + rb * lb;
            R.la = la;
            R.lb = lb;
            R.ku = inv_mag * (inv_w * inv_w);
            R.inv = __builtin_amdgcn_rcpf(nb);
            const float h = L.nlim * __builtin_fabsf(R.inv), tol = h * (8e-6f + 3e-7f * h);
            R.hm = h - tol;
            R.hp = h + tol;
            // (the walk's tangent error drifts from the exact one: a margin keeps T within [0, |t|^2])
            const float drift = L.LL * 6e-8f * (4.0f * __builtin_amdgcn_sqrtf(L.LL) + 64.0f);
            R.cap = ((L.meta & FR_SAFE) && L.nlim < 64.0f * na) ? L.cap + drift : __builtin_inff();
            R.far = L.LL - (L.cap + drift);
            R.base = ax ? (c0 - Y0) * PITCH - X0 : (c0 - X0) - Y0 * PITCH;
            R.s0 = ax ? sg.c[0] : sg.c[1];
            R.line = sg.line;
            R.meta = L.meta | (sg.ncols << 16);
            wR[lane] = R;
            if (!replay_columns<SEG>(wK, L, sg, lane * SEG, sg.ncols)) atomicOr(flags, FLAG_STUCK);
        }
        // (gaussian: after the fills, whose double exp needs the registers that the next
        // items would hold; 20 spilled ones made 100 000 lines of 1 to 8 px 211 us, now 205)
        if constexpr (K != K_GAUSSIAN) take(np);
        wave_sync();
        // phase 2a
        int ncap = 0, cap_lo = 0, cap_hi = 0;   // lane i: item i's columns in the list
        for (int u0 = 0; u0 < n * SEG; u0 += 64) {
            const int u = u0 + lane, i = u / SEG, k = u % SEG;
            bool cap = false;
            double v[3] = {0.0, 0.0, 0.0};
            if (u < n * SEG) {
                const AdjRec &R = wR[i];
                const int meta = R.meta;
                if (k < (meta >> 16)) {
                    const float Te = wK.T[u], Ne = wK.N[u];
                    const float jc = -Ne * R.inv;
                    cap = !(Te > R.cap && Te < R.far && __builtin_fabsf(jc) <= 1.0f);
                    if (!cap) {
                        const int cs = R.s0 + wK.centre(u);
                        const bool rx = meta & FR_AXIS;
                        const int kk = (meta & FR_SA) ? k : -k;
                        const int sst = rx ? 1 : PITCH;
                        const int at = R.base + kk * (rx ? PITCH : 1) + cs * sst;
                        const int w0 = (rx ? X0 : Y0) - cs, w1 = (rx ? X1 : Y1) - 1 - cs;
                        const double ra = R.la, rb = R.lb, ku = R.ku;
                        const double q0 = __builtin_fma((double)kk, rb, __builtin_fma(-(double)cs, ra, R.q0));
                        const double T0 = __builtin_fma((double)kk, ra, __builtin_fma((double)cs, rb, R.T0));
                        const float f0 = __builtin_ceilf(jc - R.hm), f1 = __builtin_floorf(jc + R.hm);
                        const int j0 = (int)f0, j1 = (int)f1;
                        const int ja = max(j0, w0), m = min(j1, w1) - ja + 1;
                        double jd = (double)ja, sums3[3] = {0.0, 0.0, 0.0};
                        const float *p = gt + (at + ja * sst);
                        for (int j = 0; j < m; j++) {
                            // (sums3[1] with j in place of T)
                            add_inside<K>(sums3, *p, __builtin_fma(-jd, ra, q0), jd, ku);
                            jd += 1.0;
                            p += sst;
                        }
                        // the undecided pixels next to the band's ends (fill_interior)
                        const float g0 = __builtin_ceilf(jc - R.hp), g1 = __builtin_floorf(jc + R.hp);
                        if (g0 < f0 || g1 > f1) {
                            const LineSetup<float> G = setup[R.line];
                            const float nb = rx ? G.nv[0] : G.nv[1];
                            for (int j = (int)g0; j <= (int)g1; j++) {
                                if ((j >= j0 && j <= j1) || j < w0 || j > w1) continue;
                                float N = Ne;
                                const float dN = (j < 0) ? -nb : nb;
                                for (int z = 0; z < abs(j); z++) N += dN;
                                if (j != 0 && !(__builtin_fabsf(N) < G.nlim)) continue;
                                if (err_fast(G, G.LL, G.ea, 0.0f, N) <= 1.0f)
                                    add_inside<K>(sums3, gt[at + j * sst], __builtin_fma(-(double)j, ra, q0), (double)j,
                                                  ku);
                            }
                        }
                        v[0] = sums3[0];
                        v[1] = __builtin_fma(T0, sums3[0], rb * sums3[1]);
                        v[2] = sums3[2];
                    }
                }
            }
            const uint64_t cm = __ballot(cap);
            if (cap) wC[ncap + __popcll(cm & below)] = (uint8_t)u;
            // the SEG lanes of one item hold its columns
#pragma unroll
            for (int j = 0; j < 3; j++) v[j] = item_sum<SEG>(v[j]);
            if (k == 0 && i < CHW)
                for (int j = 0; j < 3; j++) wX.item[i][j] = v[j];
            if (lane / IPR == u0 / 64) {
                const int from = (lane % IPR) * SEG;
                cap_lo = ncap + __popcll(cm & ((1ull << from) - 1ull));
                cap_hi = cap_lo + __popcll((cm >> from) & ((1ull << SEG) - 1ull));
            }
            ncap += __popcll(cm);
        }
        wave_sync();
        double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};   // lane i: item i's sums
        if (lane < n)
            for (int j = 0; j < 3; j++) acc[j] = wX.item[lane][j];
        // phase 2b
        for (int v0 = 0; v0 < ncap; v0 += BATCH) {
            wave_sync();
            const int v = v0 + (lane >> 1), half = lane & 1;
            double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            if (v < ncap) {
                const int slot = wC[v], i = slot / SEG, k = slot % SEG;
                const AdjRec &R = wR[i];
                const int meta = R.meta, cs = R.s0 + wK.centre(slot);
                const LineSetup<float> &G = setup[R.line];
                const bool rx = meta & FR_AXIS;
                const int kk = (meta & FR_SA) ? k : -k, sst = rx ? 1 : PITCH;
                const int at = R.base + kk * (rx ? PITCH : 1);   // (at short-axis coordinate 0)
                const int s_lo = rx ? X0 : Y0, s_hi = rx ? X1 : Y1;
                const double ra = R.la, rb = R.lb, ku = R.ku, mag = ra * ra + rb * rb;
                const double qk = __builtin_fma((double)kk, rb, R.q0), Tk = __builtin_fma((double)kk, ra, R.T0);
                auto add = [&](int s) {
                    const float p = gt[at + s * sst];
                    const double sd = (double)s;
                    if (p != 0.0f)
                        add_clamped<K>(w, p, __builtin_fma(-sd, ra, qk), __builtin_fma(sd, rb, Tk), mag, ku);
                };
                if (meta & FR_SAFE) {
                    // the centre goes with half 0
                    const float LL = G.LL, ea = G.ea, nlim = G.nlim;
                    const int sb = (meta & FR_SB) ? 1 : -1, dir = half ? -sb : sb;
                    const float tb = rx ? G.t[0] : G.t[1], nb = rx ? G.nv[0] : G.nv[1];
                    const float dT = (dir > 0) ? tb : -tb, dN = (dir > 0) ? nb : -nb;
                    float Te = wK.T[slot], Ne = wK.N[slot];
                    if (half == 0 && cs >= s_lo && cs < s_hi && err_fast(G, LL, ea, Te, Ne) <= 1.0f) add(cs);
                    const int nsteps = (dir > 0) ? (s_hi - 1 - cs) : (cs - s_lo);
                    const int jin = (dir > 0) ? (s_lo - cs) : (cs - s_hi + 1);
                    for (int j = 1; j <= nsteps; j++) {
                        Te += dT;
                        Ne += dN;
                        if (!(__builtin_fabsf(Ne) < nlim)) break;
                        if (j >= jin && err_fast(G, LL, ea, Te, Ne) <= 1.0f) add(cs + j * dir);
                    }
                } else if (half == 0) {
                    const ColRec<float> cr = {cs, wK.T[slot], wK.N[slot]};
                    fill_column(G, cr, s_lo, s_hi, [&](int s, float Te, float Ne) {
                        if (err_of(G, Te, Ne) <= 1.0f) add(s);
                    });
                }
            }
#pragma unroll
            for (int j = 0; j < 5; j++) {
                w[j] += dpp_move<0xb1>(w[j]);
                if (half == 0) wX.col[lane >> 1][j] = w[j];
            }
            wave_sync();
            for (int z = max(cap_lo, v0); z < min(cap_hi, v0 + BATCH); z++)
#pragma unroll
                for (int j = 0; j < 5; j++) acc[j] += wX.col[z - v0][j];
        }
        // the constants of the sums, and out
        if (lane < n) {
            const double mv = (double)max_val;
            double ch, cw;   // GradConst's cc, cw with the powers of |t|
            if constexpr (K == K_TRIANGULAR) {
                const double inv_len = sqrt(inv_mag);
                ch = mv * inv_w * inv_len;
                cw = mv * (inv_w * inv_w) * inv_len;
            } else {
                constexpr double kp = (K == K_BIWEIGHT) ? -1.875
                                                        : ((K == K_PARABOLIC) ? -0.75 : -4.5 * 0.3989422804014327);
                ch = -2.0 * kp * mv * (inv_w * inv_w) * inv_mag;
                cw = -2.0 * kp * mv * inv_w;
            }
            // (no product of an infinite constant with an empty sum)
            auto times = [](double c, double x) { return (x != 0.0) ? c * x : 0.0; };
            const double e1 = times(ch, acc[0]), e2 = times(ch * inv_mag, acc[1]);
            const double o1 = times(ch, acc[3]), o2 = times(ch * inv_mag, acc[4]);
            const double a1 = times(lb, e1) + times(la, o1), b1 = times(lb, o1) - times(la, e1);
            const double a2 = times(lb, e2) + times(la, o2), b2 = times(lb, o2) - times(la, e2);
            double *p = partial + 5 * out_at;
            p[0] = ax ? b1 : a1;
            p[1] = ax ? a1 : b1;
            p[2] = ax ? b2 : a2;
            p[3] = ax ? a2 : b2;
            p[4] = times(cw, acc[2]);
        }
        if (t + 1 == turns) break;   // (no items to wait for: 20 000 frames of 64^2, a line each, 195 -> 189 us)
        if constexpr (K == K_GAUSSIAN) take(np);
        wave_sync();
    }
}

// Adjoint of the double lines: one lane per column, the full terms.
template <typename T, int K, int TILE, int SEG, int NT, int CH>
__global__ void __launch_bounds__(NT)
k_adjoint_tiles(const T *__restrict__ grad, const T *__restrict__ lines, Geometry g, const int *__restrict__ tile_off,
                const int2 *__restrict__ pairs, const Segment<T> *__restrict__ segs,
                const LineSetup<T> *__restrict__ setup, const int *__restrict__ slot_base, T max_val,
                double *__restrict__ partial, int *__restrict__ flags)
{
    constexpr int NW = NT / 64;
    static_assert(64 % SEG == 0, "a segment's columns must share one round of a wave");
    __shared__ T gt[TILE * tile_pitch<TILE>()];
    __shared__ ColRec<T> rec[NW][CH * SEG];
    __shared__ ItemHdr hdr[NW][CH];

    const int tile = blockIdx.x;
    const int beg = tile_off[tile * LIST_SUBS], end = tile_off[(tile + 1) * LIST_SUBS];
    // a plan whose last draw failed (capacity, bad idxs) has no valid lists
    if (*flags || beg == end) return;
    const int per_frame = g.ntx * g.nty;
    const int64_t f = tile / per_frame;
    const int r = tile - (int)f * per_frame;
    const int ty = r / g.ntx, tx = r - ty * g.ntx;
    const int X0 = tx * TILE, Y0 = ty * TILE;
    const int X1 = min(X0 + TILE, g.W), Y1 = min(Y0 + TILE, g.H);

    const T *fg = grad + (f * g.H) * (int64_t)g.W;
    // the tile of dLoss/dImage: every load issued before the LDS writes
    static_assert((TILE * TILE) % NT == 0, "whole tile rows per thread pass");
    constexpr int PER = TILE * TILE / NT;
    T gv[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = threadIdx.x + j * NT;
        const int y = Y0 + i / TILE, x = X0 + (i % TILE);
        gv[j] = (y < Y1 && x < X1) ? __builtin_nontemporal_load(&fg[(int64_t)y * g.W + x]) : T(0);
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = threadIdx.x + j * NT;
        gt[(i / TILE) * tile_pitch<TILE>() + (i % TILE)] = gv[j];
    }
    __syncthreads();

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    ColRec<T> *R = rec[wave];
    for (int first = beg + wave * CH; first < end; first += NW * CH) {
        const int n = min(CH, end - first);
        if (lane < n) {
            const int2 it = pairs[first + lane];
            const Segment<T> sg = segs[it.x];
            const LineSetup<T> L = setup[it.y];
            hdr[wave][lane].seg = it.x;
            hdr[wave][lane].line = it.y;
            walk_columns<T, SEG>(L, sg, R, lane, flags);
        }
        wave_sync();
        const int rounds = (n * SEG + 63) / 64;
        for (int rd = 0; rd < rounds; rd++) {
            const int u = lane + 64 * rd;
            const int i = u / SEG, k = u - i * SEG;
            double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            if (i < n) {
                const ColRec<T> cr = R[u];
                if (cr.s != INT_MIN) {
                    const Segment<T> &sg = segs[hdr[wave][i].seg];
                    const LineSetup<T> &L = setup[hdr[wave][i].line];
                    const int a = L.axis;
                    const int c = pick(sg.c, a) + k * pick(L.st, a);
                    const int s_lo = (a == 0) ? Y0 : X0, s_hi = (a == 0) ? Y1 : X1;
                    const GradConst C = grad_const<K>(L, lines + 5 * (int64_t)hdr[wave][i].line, max_val);
                    fill_column(L, cr, s_lo, s_hi, [&](int s, T Te, T Ne) {
                        const T err = err_of(L, Te, Ne);
                        if (!(err <= T(1))) return;
                        const int x = (a == 0) ? c : s, y = (a == 0) ? s : c;
                        const T gv = gt[(y - Y0) * tile_pitch<TILE>() + (x - X0)];
                        if (gv != T(0)) pixel_grad<K>(C, x, y, (double)gv, acc);
                    });
                }
            }
            // the SEG lanes of one item hold its columns: reduce them in a fixed tree
#pragma unroll
            for (int m = SEG / 2; m > 0; m >>= 1)
#pragma unroll
                for (int j = 0; j < 5; j++) acc[j] += __shfl_xor(acc[j], m, SEG);
            if (k == 0 && i < n) {
                const int sid = hdr[wave][i].seg;
                const Segment<T> &sg = segs[sid];
                const int a = setup[hdr[wave][i].line].axis;
                const int tb = (a == 0) ? ty : tx;
                double *p = partial + 5 * (int64_t)(slot_base[sid] + (tb - (sg.lo >> g.tile_log)));
#pragma unroll
                for (int j = 0; j < 5; j++) p[j] = acc[j];
            }
        }
        wave_sync();
    }
}

// Per-line sums of the partials (deterministic): LG_LANES lanes per line,
// lane j adding the line's partials j, j + LG_LANES, ... in slot order, then a
// fixed butterfly over the lanes.  A line's slots are [line_base[l],
// line_base[l] + segment_bound); slot s's partials start at slot_base[s].
constexpr int LG_LANES = 8;

template <typename T>
__global__ void __launch_bounds__(256)
k_line_grad(const int64_t *__restrict__ line_base, const LineSetup<T> *__restrict__ setup, Geometry g,
            const int *__restrict__ slot_base, const double *__restrict__ partial, int64_t n_lines,
            T *__restrict__ grad_lines, const int *__restrict__ flags)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t l = t / LG_LANES;
    const int j = (int)(t % LG_LANES);
    // after a failed draw of a plan the slot ranges are not valid (the
    // gradient stays zero; the error is reported by the plan's check)
    const bool ok = l < n_lines && *flags == 0;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (ok) {
        const int ub = segment_bound(setup[l], g);
        const int64_t s0 = slot_base[line_base[l]], s1 = slot_base[line_base[l] + ub];
        for (int64_t s = s0 + j; s < s1; s += LG_LANES)
#pragma unroll
            for (int k = 0; k < 5; k++) acc[k] += partial[5 * s + k];
    }
#pragma unroll
    for (int m = LG_LANES / 2; m > 0; m >>= 1)
#pragma unroll
        for (int k = 0; k < 5; k++) acc[k] += __shfl_xor(acc[k], m, LG_LANES);
    if (!ok || j != 0) return;
    // (sum c dx - sum c ts dx, ..., sum c ts dx, ...): see pixel_grad
    grad_lines[5 * l + 0] = (T)(acc[0] - acc[2]);
    grad_lines[5 * l + 1] = (T)(acc[1] - acc[3]);
    grad_lines[5 * l + 2] = (T)acc[2];
    grad_lines[5 * l + 3] = (T)acc[3];
    grad_lines[5 * l + 4] = (T)acc[4];
}

// ---------------------------------------------------------------------------
// host pipeline
// ---------------------------------------------------------------------------
static int check_common(int64_t n_frames, int64_t H, int64_t W, int64_t n_lines, bool have_idxs, int kernel,
                        int overlap)
{
    if (kernel < 0 || kernel > 4) return fail(CBX_EVALUE, "kernel is missing for id " + std::to_string(kernel));
    if (overlap < 0 || overlap > 1) return fail(CBX_EVALUE, "Invalid overlap keyword");
    if (n_frames < 0 || H < 0 || W < 0 || n_lines < 0) return fail(CBX_EVALUE, "negative size");
    if (H > (1 << 30) || W > (1 << 30) || n_frames >= (int64_t(1) << 31))
        return fail(CBX_EVALUE, "frame shape exceeds the supported range");
    if (n_lines >= (int64_t(1) << 31)) return fail(CBX_EVALUE, "too many lines");
    if (!have_idxs && n_lines && n_frames != 1 && n_frames != n_lines)
        return fail(CBX_EVALUE, "idxs has an incompatible size (" + std::to_string(n_lines) +
                                    " != " + std::to_string(n_frames) + ")");
    return CBX_OK;
}

static int flags_to_status(int flags)
{
    if (flags & FLAG_INDEX) return fail(CBX_EINDEX, "idxs is outside of (0, n_frames)");
    if (flags & FLAG_LONG)
        return fail(CBX_EVALUE, "a line's walk exceeds the supported length (2^26 px) or coordinate range (1e9)");
    if (flags & FLAG_KERNEL) return fail(CBX_EVALUE, "kernel is missing for a per-line profile id");
    if (flags & FLAG_STUCK) return fail(CBX_ERUNTIME, "a line walk did not terminate within its step budget");
    if (flags & FLAG_OVERFLOW) return fail(CBX_ECAPACITY, "the plan's segment or tile-item capacity was exceeded");
    return CBX_OK;
}

// Builds segments (and, with bin, the per-tile item lists).  One host sync.
template <typename T, typename I>
static int build_plan(SegmentPlan<T> &P, const T *lines, const I *idxs, int kernel, int64_t n_lines,
                      int64_t n_frames, int64_t H, int64_t W, int tile, int seg, bool bin, hipStream_t st,
                      bool skip_neg = false)
{
    Geometry &g = P.g;
    g.skip_neg = skip_neg ? 1 : 0;
    g.n_frames = n_frames;
    g.H = (int32_t)H;
    g.W = (int32_t)W;
    set_tiles(g, tile, seg);
    P.n_lines = n_lines;
    P.n_tiles = bin ? n_frames * g.ntx * g.nty : 0;
    if (P.n_tiles >= (int64_t(1) << 31)) return fail(CBX_EVALUE, "too many tiles");

    CBX_HIP(P.setup.alloc(n_lines, st));
    CBX_HIP(P.seg_cnt.alloc(n_lines + 1, st));
    CBX_HIP(P.seg_off.alloc(n_lines + 1, st));
    CBX_HIP(P.flags.alloc(1, st));
    CBX_HIP(hipMemsetAsync(P.flags.ptr, 0, sizeof(int), st));
    CBX_HIP(hipMemsetAsync(P.seg_cnt.ptr + n_lines, 0, sizeof(int), st));
    if (bin) {
        CBX_HIP(P.tile_cnt.alloc(P.n_tiles + 1, st));
        CBX_HIP(P.tile_off.alloc(P.n_tiles + 1, st));
        CBX_HIP(hipMemsetAsync(P.tile_cnt.ptr, 0, sizeof(int) * (P.n_tiles + 1), st));
    }
    const int blk = 256;
    {
        KernelTimer timer1("segments_pass1", st);
    if (bin)
        k_segments<T, I, false, true><<<grid_for(n_lines, blk), blk, 0, st>>>(
            lines, idxs, kernel, n_lines, g, P.setup.ptr, P.seg_cnt.ptr, P.tile_cnt.ptr, nullptr, nullptr, nullptr, nullptr,
            nullptr, P.flags.ptr);
    else
        k_segments<T, I, false, false><<<grid_for(n_lines, blk), blk, 0, st>>>(
            lines, idxs, kernel, n_lines, g, P.setup.ptr, P.seg_cnt.ptr, nullptr, nullptr, nullptr, nullptr, nullptr,
            nullptr, P.flags.ptr);
    }
    CBX_HIP(hipGetLastError());
    CBX_HIP(exclusive_scan_i32(P.seg_cnt.ptr, P.seg_off.ptr, n_lines + 1, st));
    if (bin) CBX_HIP(exclusive_scan_i32(P.tile_cnt.ptr, P.tile_off.ptr, P.n_tiles + 1, st));

    int host[3] = {0, 0, 0};
    {
        const void *src[3] = {P.flags.ptr, P.seg_off.ptr + n_lines, bin ? (const void *)(P.tile_off.ptr + P.n_tiles)
                                                                         : (const void *)P.flags.ptr};
        const int nb[3] = {4, 4, 4};
        uint64_t hv[3];
        CBX_HIP(read_device_values(st, 3, src, nb, hv));
        for (int i = 0; i < 3; i++) host[i] = (int)(uint32_t)hv[i];
        if (!bin) host[2] = 0;
    }
    int rc = flags_to_status(host[0]);
    if (rc) return rc;
    if (host[1] < 0 || host[2] < 0) return fail(CBX_ERUNTIME, "segment count overflow");
    P.n_segs = host[1];
    P.n_items = host[2];
    if (P.n_segs == 0) return CBX_OK;

    CBX_HIP(P.segs.alloc(P.n_segs, st));
    if (bin) {
        CBX_HIP(P.items.alloc(P.n_items, st));
        CBX_HIP(P.tile_cur.alloc(P.n_tiles, st));
        CBX_HIP(hipMemsetAsync(P.tile_cur.ptr, 0, sizeof(int) * P.n_tiles, st));
        k_segments<T, I, true, true><<<grid_for(n_lines, blk), blk, 0, st>>>(
            lines, idxs, kernel, n_lines, g, P.setup.ptr, nullptr, nullptr, P.seg_off.ptr, P.segs.ptr, P.tile_off.ptr,
            P.tile_cur.ptr, P.items.ptr, P.flags.ptr);
    } else {
        k_segments<T, I, true, false><<<grid_for(n_lines, blk), blk, 0, st>>>(
            lines, idxs, kernel, n_lines, g, P.setup.ptr, nullptr, nullptr, P.seg_off.ptr, P.segs.ptr, nullptr, nullptr,
            nullptr, P.flags.ptr);
    }
    CBX_HIP(hipGetLastError());
    return CBX_OK;
}

// Largest slot total of the eager unordered plans so far (a capacity hint
// for the next).
static std::atomic<int64_t> g_slot_hint{0};

// Unordered plan for the tile path: one walk per line (k_setup_lines,
// k_walk_lines, k_bin_slots).  Segments live in slots (n_segs = slots; unused
// slots have ncols = 0 and are in no item list).  One host read after the
// walk (the item total, flags, the slot total), one more before it when the
// previous call's slot total is no usable capacity.
template <typename T, typename I>
static int build_plan_unordered(SegmentPlan<T> &P, const T *lines, const I *idxs, const uint8_t *kernels,
                                int kernel, int64_t n_lines, int64_t n_frames, int64_t H, int64_t W, int tile,
                                int seg, hipStream_t st, int64_t *line_base = nullptr, bool slot_tiles = false, bool skip_neg = false)
{
    Geometry &g = P.g;
    g.skip_neg = skip_neg ? 1 : 0;
    g.n_frames = n_frames;
    g.H = (int32_t)H;
    g.W = (int32_t)W;
    set_tiles(g, tile, seg);
    P.n_lines = n_lines;
    P.n_tiles = n_frames * g.ntx * g.nty;
    if (P.n_tiles >= (int64_t(1) << 31) / LIST_SUBS) return fail(CBX_EVALUE, "too many tiles");
    const int64_t n_lists = P.n_tiles * LIST_SUBS;

    DevBuf<unsigned long long> counters;
    CBX_HIP(P.setup.alloc(n_lines, st));
    if (sizeof(T) == 4) CBX_HIP(P.lite.alloc(n_lines, st));
    CBX_HIP(P.flags.alloc(1, st));
    CBX_HIP(counters.alloc(2, st));
    CBX_HIP(P.tile_cnt.alloc(n_lists, st));
    CBX_HIP(P.tile_off.alloc(n_lists + 1, st));
    CBX_HIP(P.tile_cur.alloc(n_lists, st));
    {
        // every counter of the pass, cleared by one kernel
        void *const zp[4] = {P.flags.ptr, counters.ptr, P.tile_cnt.ptr, P.tile_cur.ptr};
        const int64_t zw[4] = {1, 4, n_lists, n_lists};
        CBX_HIP(zero_words(st, 4, zp, zw));
    }
    const int blk = 256;
    k_setup_lines<T, I><<<grid_for(n_lines, blk), blk, 0, st>>>(lines, idxs, kernels, kernel, n_lines, g,
                                                               P.setup.ptr, P.lite.ptr, counters.ptr, P.flags.ptr);
    CBX_HIP(hipGetLastError());
    uint64_t hv[3];
    int fl = 0, rc = 0;
    // Slot capacity: the largest slot total of the previous calls when it is
    // not far above what these lines could need, so the walk starts without
    // reading this call's total first; a walk that runs out of slots
    // (FLAG_OVERFLOW with a larger total) is cleared and run again at the
    // exact total.  Without a usable hint the total is read first.
    int64_t cap = g_slot_hint.load(std::memory_order_relaxed);
    if (cap <= 0 || cap > 64 * n_lines + 65536) {
        const void *src[2] = {counters.ptr, P.flags.ptr};
        const int nb[2] = {8, 4};
        CBX_HIP(read_device_values(st, 2, src, nb, hv));
        fl = (int)(uint32_t)hv[1];
        if ((rc = flags_to_status(fl))) return rc;
        if (hv[0] >= (1ull << 31)) return fail(CBX_EVALUE, "too many segments (2^31)");
        cap = (int64_t)hv[0];
        if (cap == 0) {
            P.n_segs = 0;
            return CBX_OK;
        }
    }
    int64_t slots = 0;
    for (int attempt = 0;; attempt++) {
        CBX_HIP(P.segs.alloc(cap, st));
        {
            KernelTimer timer("segments_walk", st);
            k_walk_lines<T><<<grid_for(n_lines, blk), blk, 0, st>>>(n_lines, g, P.setup.ptr, P.segs.ptr, cap,
                                                                    counters.ptr, P.tile_cnt.ptr, P.flags.ptr,
                                                                    line_base);
        }
        CBX_HIP(hipGetLastError());
        // list offsets (tile_off[n_lists]: the item total)
        CBX_HIP(exclusive_scan_total_i32(P.tile_cnt.ptr, nullptr, P.tile_off.ptr, n_lists, st));
        {
            const void *src[3] = {P.tile_off.ptr + n_lists, P.flags.ptr, counters.ptr};
            const int nb[3] = {4, 4, 8};
            CBX_HIP(read_device_values(st, 3, src, nb, hv));
        }
        fl = (int)(uint32_t)hv[1];
        if ((rc = flags_to_status(fl & ~FLAG_OVERFLOW))) return rc;
        if (hv[2] >= (1ull << 31)) return fail(CBX_EVALUE, "too many segments (2^31)");
        slots = (int64_t)hv[2];
        if (!(fl & FLAG_OVERFLOW)) break;
        if (attempt > 0 || slots <= cap) return flags_to_status(fl);   // cannot happen: the total fits
        // too few slots: clear what the walk counted and walk again
        cap = slots;
        void *const zp[4] = {P.flags.ptr, counters.ptr + 1, P.tile_cnt.ptr, P.tile_cur.ptr};
        const int64_t zw[4] = {1, 2, n_lists, n_lists};
        CBX_HIP(zero_words(st, 4, zp, zw));
    }
    // the largest total so far: calls of varying sizes rarely walk twice
    for (int64_t h = g_slot_hint.load(std::memory_order_relaxed);
         h < slots && !g_slot_hint.compare_exchange_weak(h, slots, std::memory_order_relaxed);) {
    }
    P.n_segs = slots;
    if (P.n_segs == 0) return CBX_OK;
    const int n_items = (int)(uint32_t)hv[0];
    if (n_items < 0) return fail(CBX_ERUNTIME, "tile item count overflow");
    P.n_items = n_items;
    CBX_HIP(P.pairs.alloc(P.n_items, st));
    if (slot_tiles) CBX_HIP(P.slot_tiles.alloc(P.n_segs, st));
    k_bin_slots<T><<<grid_for(P.n_segs, blk), blk, 0, st>>>(P.n_segs, g, P.setup.ptr, P.segs.ptr, P.tile_off.ptr,
                                                            P.tile_cur.ptr, P.pairs.ptr, counters.ptr, P.n_tiles,
                                                            P.n_items, P.flags.ptr, P.slot_tiles.ptr);
    CBX_HIP(hipGetLastError());
    return CBX_OK;
}

// Tile and segment size where the caller names none: 64 x 64 tiles with a
// checkpoint every 8 columns are the fastest shape of many tiles (64 frames of
// 2048^2), but a workgroup per tile leaves CUs idle where the frames have no more
// tiles than the card has CUs (256); there tiles of 32 x 32 share the work of a
// tile among four workgroups.  Measured for 64 / 32, us: doubles 154 / 114 at 64
// tiles, 161 / 131 at 256; gradients 170 / 148 at 64, 178 / 163 at 256, 136 / 140 at
// 704; float draws 79 / 61 with 5000 lines in 64 tiles, 118 / 114 with 1000, and
// where a tile has a few lines only 75 / 78 (192 lines in 64 tiles, gradient 102 / 101).
// A frame of at most 32 x 32 is one tile either way, of which less is cleared, read and
// written (20 000 frames of 16^2, a line each: 108 / 82, gradient 164 / 153).
// The frames decide, not the lines or the pass, so that a plan, the eager draw and the
// eager gradient of the same frames work on the same tiles and give the same bits.
static void resolve_opts(const cbx_draw_opts *o, int64_t n_frames, int64_t H, int64_t W, int &tile, int &seg)
{
    const double tiles = (double)n_frames * (double)((H + 63) / 64) * (double)((W + 63) / 64);
    tile = (o && o->tile) ? o->tile : ((tiles <= 256.0 || (H <= 32 && W <= 32)) ? 32 : 64);
    seg = (o && o->seg) ? o->seg : 8;
}

static int check_opts(int tile, int seg)
{
    if (!(tile == 32 || tile == 64)) return fail(CBX_EVALUE, "tile must be 32 or 64");
    if (!(seg == 8 || seg == 16)) return fail(CBX_EVALUE, "seg must be 8 or 16");
    return CBX_OK;
}

template <typename T, bool WRITE>
static void launch_emit(int kernel, const SegmentPlan<T> &P, T max_val, int *cnt, const int64_t *off,
                        uint64_t *keys, T *vals, int32_t *lines_out, hipStream_t st)
{
    const int blk = 256;
    const int grid = grid_for(P.n_segs, blk);
#define CBX_EMIT(KK)                                                                                           \
    k_emit<T, KK, WRITE><<<grid, blk, 0, st>>>(P.segs.ptr, P.n_segs, P.setup.ptr, P.g.H, P.g.W, max_val, cnt, off, \
                                              keys, vals, lines_out, P.flags.ptr)
    switch (kernel) {
    case K_BIWEIGHT: CBX_EMIT(K_BIWEIGHT); break;
    case K_GAUSSIAN: CBX_EMIT(K_GAUSSIAN); break;
    case K_PARABOLIC: CBX_EMIT(K_PARABOLIC); break;
    case K_RECTANGULAR: CBX_EMIT(K_RECTANGULAR); break;
    default: CBX_EMIT(K_TRIANGULAR); break;
    }
#undef CBX_EMIT
}

// Raw pixel list: one entry per emitted pixel, in the reference's emission
// order (segments are stored line-major, in walk order).
template <typename T>
static int raw_list_pipeline(SegmentPlan<T> &P, int kernel, T max_val, int32_t *of, int32_t *oy, int32_t *ox, T *ov,
                             int32_t *ol, int64_t capacity, int64_t *count, hipStream_t st)
{
    *count = 0;
    if (P.n_segs == 0) return CBX_OK;
    const int blk = 256;
    DevBuf<int> cnt;
    DevBuf<int64_t> cnt64, off;
    CBX_HIP(cnt.alloc(P.n_segs + 1, st));
    CBX_HIP(cnt64.alloc(P.n_segs + 1, st));
    CBX_HIP(off.alloc(P.n_segs + 1, st));
    CBX_HIP(hipMemsetAsync(cnt.ptr + P.n_segs, 0, sizeof(int), st));
    launch_emit<T, false>(kernel, P, max_val, cnt.ptr, nullptr, nullptr, nullptr, nullptr, st);
    CBX_HIP(hipGetLastError());
    k_i32_to_i64<<<grid_for(P.n_segs + 1, blk), blk, 0, st>>>(cnt.ptr, cnt64.ptr, P.n_segs + 1);
    CBX_HIP(exclusive_scan_i64(cnt64.ptr, off.ptr, P.n_segs + 1, st));
    int64_t E = 0;
    int fl = 0;
    {
        const void *src[2] = {off.ptr + P.n_segs, P.flags.ptr};
        const int nb[2] = {8, 4};
        uint64_t hv[2];
        CBX_HIP(read_device_values(st, 2, src, nb, hv));
        E = (int64_t)hv[0];
        fl = (int)(uint32_t)hv[1];
    }
    int rc = flags_to_status(fl);
    if (rc) return rc;
    *count = E;
    if (E == 0 || E > capacity) return CBX_OK;
    DevBuf<uint64_t> keys;
    DevBuf<T> vals;
    DevBuf<int32_t> lof;
    CBX_HIP(keys.alloc(E, st));
    CBX_HIP(vals.alloc(E, st));
    const bool want_lines = (ol != nullptr);
    if (want_lines) CBX_HIP(lof.alloc(E, st));
    launch_emit<T, true>(kernel, P, max_val, nullptr, off.ptr, keys.ptr, vals.ptr, want_lines ? lof.ptr : nullptr,
                         st);
    CBX_HIP(hipGetLastError());
    k_raw_out<T><<<grid_for(E, blk), blk, 0, st>>>(keys.ptr, vals.ptr, lof.ptr, E, P.g.H, P.g.W, of, oy, ox, ov,
                                                  want_lines ? ol : nullptr);
    CBX_HIP(hipGetLastError());
    CBX_HIP(hipStreamSynchronize(st));
    return CBX_OK;
}

// tile_list = nullptr: one workgroup per plan tile; otherwise one per entry of
// tile_list (n_list tile ids).
template <typename T, int OV, int TILE, int SEG, bool LIST, int ACC = -1>
static void launch_ordered_k(int kernel, T *img, uint8_t *touched, int32_t *first, const SegmentPlan<T> &P,
                             T max_val, hipStream_t st, const int32_t *term_frame = nullptr,
                             const int *tile_list = nullptr, int64_t n_list = 0)
{
    const unsigned grid = (unsigned)(tile_list ? n_list : P.n_tiles);
#define CBX_ORD(KK)                                                                                             \
    k_tiles_ordered<T, KK, OV, TILE, SEG, LIST, ACC><<<grid, 64, 0, st>>>(                                      \
        img, touched, first, P.g, P.tile_off.ptr, P.items.ptr, P.segs.ptr, P.setup.ptr, max_val, P.flags.ptr,    \
        term_frame, tile_list)
    switch (kernel) {
    case K_BIWEIGHT: CBX_ORD(K_BIWEIGHT); break;
    case K_GAUSSIAN: CBX_ORD(K_GAUSSIAN); break;
    case K_PARABOLIC: CBX_ORD(K_PARABOLIC); break;
    case K_RECTANGULAR: CBX_ORD(K_RECTANGULAR); break;
    default: CBX_ORD(K_TRIANGULAR); break;
    }
#undef CBX_ORD
}

// Reference-order accumulation over a binned plan (tile 32, seg 16):
// image != nullptr accumulates into the caller's frames; otherwise a merged
// pixel list is compacted out of a dense scratch render.
template <typename T>
static int ordered_pipeline(SegmentPlan<T> &P, int kernel, int overlap, T max_val, T *image, int32_t *of, int32_t *oy,
                            int32_t *ox, T *ov, int32_t *ol, int64_t capacity, int64_t *count, hipStream_t st)
{
    if (count) *count = 0;
    if (P.n_segs == 0) return CBX_OK;
    k_sort_tile_items<<<(unsigned)P.n_tiles, 256, 0, st>>>(P.tile_off.ptr, P.items.ptr, P.flags.ptr, nullptr);
    CBX_HIP(hipGetLastError());
    const int64_t npix = P.g.n_frames * (int64_t)P.g.H * P.g.W;
    DevBuf<T> scratch;
    DevBuf<uint8_t> touched;
    DevBuf<int32_t> first;
    T *img = image;
    if (!image) {
        CBX_HIP(scratch.alloc(npix, st));
        CBX_HIP(touched.alloc(npix, st));
        if (ol) CBX_HIP(first.alloc(npix, st));
        // tiles without items never write their flags
        CBX_HIP(hipMemsetAsync(touched.ptr, 0, npix, st));
        img = scratch.ptr;
    }
    if (overlap == 0) {
        if (image) launch_ordered_k<T, 0, 32, 16, false>(kernel, img, nullptr, nullptr, P, max_val, st);
        else launch_ordered_k<T, 0, 32, 16, true>(kernel, img, touched.ptr, first.ptr, P, max_val, st);
    } else {
        if (image) launch_ordered_k<T, 1, 32, 16, false>(kernel, img, nullptr, nullptr, P, max_val, st);
        else launch_ordered_k<T, 1, 32, 16, true>(kernel, img, touched.ptr, first.ptr, P, max_val, st);
    }
    CBX_HIP(hipGetLastError());
    int fl = 0;
    {
        const void *src[1] = {P.flags.ptr};
        const int nb[1] = {4};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        fl = (int)(uint32_t)hv;
    }
    if (fl & FLAG_TILE_FULL)
        return fail(CBX_ERUNTIME, "a tile holds more than 8192 segments; the ordered mode cannot sort it");
    int rc = flags_to_status(fl);
    if (rc || image) return rc;

    const int blk = 256;
    const int64_t rows = P.g.n_frames * (int64_t)P.g.H;
    DevBuf<int64_t> rcnt, roff;
    CBX_HIP(rcnt.alloc(rows + 1, st));
    CBX_HIP(roff.alloc(rows + 1, st));
    CBX_HIP(hipMemsetAsync(rcnt.ptr + rows, 0, sizeof(int64_t), st));
    k_row_count<<<grid_for(rows, blk), blk, 0, st>>>(touched.ptr, rows, P.g.W, rcnt.ptr);
    CBX_HIP(exclusive_scan_i64(rcnt.ptr, roff.ptr, rows + 1, st));
    int64_t U = 0;
    {
        const void *src[1] = {roff.ptr + rows};
        const int nb[1] = {8};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        U = (int64_t)hv;
    }
    *count = U;
    if (U == 0 || U > capacity) return CBX_OK;
    k_row_write<T><<<grid_for(rows, blk), blk, 0, st>>>(touched.ptr, img, first.ptr, rows, P.g.H, P.g.W, roff.ptr, of,
                                                       oy, ox, ov, ol);
    CBX_HIP(hipGetLastError());
    CBX_HIP(hipStreamSynchronize(st));
    return CBX_OK;
}

// The tile kernel over a built unordered plan; kernel may be K_MIXED.
template <typename T>
static void run_tiles(T *out, const SegmentPlan<T> &P, int kernel, int overlap, T max_val, const cbx_draw_opts *opts,
                      hipStream_t st)
{
    switch (kernel) {
    case K_BIWEIGHT: run_tiles_profile<T, K_BIWEIGHT>(out, P, max_val, overlap, opts, st); break;
    case K_GAUSSIAN: run_tiles_profile<T, K_GAUSSIAN>(out, P, max_val, overlap, opts, st); break;
    case K_PARABOLIC: run_tiles_profile<T, K_PARABOLIC>(out, P, max_val, overlap, opts, st); break;
    case K_RECTANGULAR: run_tiles_profile<T, K_RECTANGULAR>(out, P, max_val, overlap, opts, st); break;
    case K_TRIANGULAR: run_tiles_profile<T, K_TRIANGULAR>(out, P, max_val, overlap, opts, st); break;
    default: run_tiles_profile<T, K_MIXED>(out, P, max_val, overlap, opts, st); break;
    }
}

template <typename T, typename I>
static int draw_lines_impl(T *out, int64_t n_frames, int64_t H, int64_t W, const T *lines, int64_t n_lines,
                           const I *idxs, T max_val, int kernel, int overlap, const cbx_draw_opts *opts, void *stream)
{
    int rc = check_common(n_frames, H, W, n_lines, idxs != nullptr, kernel, overlap);
    if (rc) return rc;
    int tile, seg;
    resolve_opts(opts, n_frames, H, W, tile, seg);
    if ((rc = check_opts(tile, seg))) return rc;
    if (opts && !(opts->threads == 0 || opts->threads == 64 || opts->threads == 128 || opts->threads == 256))
        return fail(CBX_EVALUE, "threads must be 64, 128 or 256");
    if (n_lines == 0 || n_frames * H * W == 0) return CBX_OK;
    hipStream_t st = (hipStream_t)stream;
    const bool det = opts && opts->deterministic;
    const uint8_t *kernels = opts ? opts->kernels : nullptr;
    if (kernels && det) return fail(CBX_EVALUE, "per-line profiles are drawn by the tile path only (deterministic = 0)");
    if (det) {
        tile = 32;
        seg = 16;
    }
    SegmentPlan<T> P;
    // `out` may become ready on another stream: wait for it only before the
    // first kernel that touches it
    const hipEvent_t out_ready = opts ? (hipEvent_t)opts->out_ready : nullptr;
    if (det) {
        if ((rc = build_plan<T, I>(P, lines, idxs, kernel, n_lines, n_frames, H, W, tile, seg, true, st))) return rc;
        if (out_ready) CBX_HIP(hipStreamWaitEvent(st, out_ready, 0));
        if (P.n_segs == 0) return CBX_OK;
        return ordered_pipeline<T>(P, kernel, overlap, max_val, out, nullptr, nullptr, nullptr, nullptr, nullptr, 0,
                                   nullptr, st);
    }
    if ((rc = build_plan_unordered<T, I>(P, lines, idxs, kernels, kernel, n_lines, n_frames, H, W, tile, seg, st)))
        return rc;
    if (out_ready) CBX_HIP(hipStreamWaitEvent(st, out_ready, 0));
    if (P.n_segs == 0) return CBX_OK;
    {
        KernelTimer timer("draw_tiles", st);
        run_tiles<T>(out, P, kernels ? K_MIXED : kernel, overlap, max_val, opts, st);
    }
    CBX_HIP(hipGetLastError());
    return CBX_OK;
}

template <typename T, typename I>
static int draw_pixels_impl(int64_t n_frames, int64_t H, int64_t W, const T *lines, int64_t n_lines, const I *idxs,
                            T max_val, int kernel, int overlap, int merge, int32_t *of, int32_t *oy, int32_t *ox,
                            T *ov, int32_t *ol, int64_t capacity, int64_t *count, void *stream)
{
    if (!count) return fail(CBX_EVALUE, "count must not be NULL");
    *count = 0;
    int rc = check_common(n_frames, H, W, n_lines, idxs != nullptr, kernel, overlap);
    if (rc) return rc;
    if (n_lines == 0 || n_frames * H * W == 0) return CBX_OK;
    hipStream_t st = (hipStream_t)stream;
    SegmentPlan<T> P;
    if ((rc = build_plan<T, I>(P, lines, idxs, kernel, n_lines, n_frames, H, W, 32, 16, merge != 0, st))) return rc;
    if (merge) return ordered_pipeline<T>(P, kernel, overlap, max_val, nullptr, of, oy, ox, ov, ol, capacity, count, st);
    return raw_list_pipeline<T>(P, kernel, max_val, of, oy, ox, ov, ol, capacity, count, st);
}

// accumulate_lines, step 1: range checks of terms and frames (bad[0]: a term
// outside [0, n_terms), bad[1]: a frame outside [0, n_frames)), the frame of
// every term as int32 (frames32, n_terms entries) and, when comp != nullptr,
// the frame of every line, comp[i] = frames[terms[i]].
template <typename I>
__global__ void k_term_frames(const I *__restrict__ terms, const I *__restrict__ frames, int64_t n_lines,
                              int64_t n_terms, int64_t n_frames, I *__restrict__ comp,
                              int32_t *__restrict__ frames32, int *__restrict__ bad)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n_terms) {
        const I f = frames[i];
        const bool ok = f >= 0 && (int64_t)f < n_frames;
        if (!ok) atomicOr(bad + 1, 1);
        frames32[i] = ok ? (int32_t)f : 0;
    }
    if (i < n_lines) {
        const I t = terms[i];
        I f = 0;
        if (t < 0 || (int64_t)t >= n_terms) atomicOr(bad, 1);
        else f = frames[t];
        if (comp) comp[i] = (f < 0 || (int64_t)f >= n_frames) ? I(0) : f;
    }
}

// Lines of every term (cnt) and each line's place among them (rank, in no fixed
// order), unless a term has more than `most` lines: then *many is set, counting
// stops and what was counted is of no use.  The lines of one term in a wave take one
// atomic.  Counters of few long terms share a cache line, whose atomics take 11 ns
// each one after the other (300 000 shuffled lines of 20 terms, an atomic each:
// 3.3 ms), so few workgroups run at a time and see what the ones before have found.
constexpr int TERM_COUNT_BLOCKS = 64;

template <typename I>
__global__ void __launch_bounds__(256)
k_term_count(const I *__restrict__ terms, int64_t n_lines, int64_t n_terms, int most, int *__restrict__ cnt,
             int *__restrict__ rank, int *__restrict__ many)
{
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    for (int64_t i0 = blockIdx.x * (int64_t)256 + (threadIdx.x & ~63); i0 < n_lines; i0 += gridDim.x * (int64_t)256) {
        const int64_t i = i0 + lane;
        const int64_t t64 = (i < n_lines) ? (int64_t)terms[i] : -1;
        if (__hip_atomic_load(many, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
        const bool ok = t64 >= 0 && t64 < n_terms;   // (others: k_term_frames)
        const int t = ok ? (int)t64 : -1;
        int lead = lane, place = 0, n = 0;
        for (uint64_t rest = __ballot(ok); rest;) {
            const int l = __builtin_ctzll(rest);
            const uint64_t m = __ballot(t == __shfl(t, l, 64));
            if ((m >> lane) & 1) {
                lead = l;
                place = __popcll(m & below);
                n = __popcll(m);
            }
            rest &= ~m;
        }
        int base = 0;
        if (ok && lead == lane) {
            base = atomicAdd(&cnt[t], n);
            if (base + n > most) atomicOr(many, 1);
        }
        base = __shfl(base, lead, 64);
        if (ok) rank[i] = base + place;
    }
}

// lines by term: order[off[t] + rank[i]] = i
template <typename I>
__global__ void k_term_order(const I *__restrict__ terms, const int *__restrict__ off, const int *__restrict__ rank,
                             int64_t n_lines, int *__restrict__ order)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n_lines) order[off[terms[i]] + rank[i]] = (int)i;
}

// Squared distance of point (px, py) to the segment (ax, ay)-(bx, by).
__device__ __forceinline__ double point_segment2(double px, double py, double ax, double ay, double bx, double by)
{
    const double ux = bx - ax, uy = by - ay, m = ux * ux + uy * uy;
    double t = (m > 0.0) ? ((px - ax) * ux + (py - ay) * uy) / m : 0.0;
    t = fmin(fmax(t, 0.0), 1.0);
    const double dx = px - ax - t * ux, dy = py - ay - t * uy;
    return dx * dx + dy * dy;
}

// Splits the lines: one that another line of its term may touch (draw a pixel of)
// keeps its term in `touching` and gets frame -1, one alone in its pixels gets
// -1 in `touching` and keeps its frame; *n_touching counts the former.  Every pixel
// of a line lies within its width of the segment, up to the drift of the float
// walk: lines further apart than both widths, 1 px, 1e-4 of their lengths and 2^-23
// of the squares of lengths and widths share none.  (The errors' running sums reach
// length^2 along the line, and width x length in a fill; each of as many additions as
// there are pixels rounds them by at most 2^-24, and a pixel is `length` of them.)
// (A line that draws nothing, e.g. a NaN end point, touches none.)
template <typename T, typename I>
__global__ void __launch_bounds__(256)
k_term_touch(const T *__restrict__ lines, const I *__restrict__ terms, const int *__restrict__ off,
             const int *__restrict__ order, int64_t n_lines, I *__restrict__ frame, I *__restrict__ touching,
             int *__restrict__ n_touching)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    bool touch = false;
    if (i < n_lines) {
        const int t = (int)terms[i];
        const T *a = lines + 5 * i;
        const double ax = a[0], ay = a[1], bx = a[2], by = a[3], wa = a[4];
        const double la = fabs(bx - ax) + fabs(by - ay);
        for (int k = off[t]; k < off[t + 1] && !touch; k++) {
            const int j = order[k];
            if (j == (int)i) continue;
            const T *b = lines + 5 * (int64_t)j;
            const double cx = b[0], cy = b[1], dx = b[2], dy = b[3];
            const double lb = fabs(dx - cx) + fabs(dy - cy), ws = wa + (double)b[4];
            const double r = ws + 1.0 + 1e-4 * (la + lb) + 1.2e-7 * (la * la + lb * lb + ws * ws);
            if (!(fmax(cx, dx) + r >= fmin(ax, bx) && fmin(cx, dx) - r <= fmax(ax, bx) &&
                  fmax(cy, dy) + r >= fmin(ay, by) && fmin(cy, dy) - r <= fmax(ay, by)))
                continue;
            // the segments cross, or the distance is an end point's
            const double o1 = (bx - ax) * (cy - ay) - (by - ay) * (cx - ax);
            const double o2 = (bx - ax) * (dy - ay) - (by - ay) * (dx - ax);
            const double o3 = (dx - cx) * (ay - cy) - (dy - cy) * (ax - cx);
            const double o4 = (dx - cx) * (by - cy) - (dy - cy) * (bx - cx);
            const double d2 = fmin(fmin(point_segment2(ax, ay, cx, cy, dx, dy), point_segment2(bx, by, cx, cy, dx, dy)),
                                   fmin(point_segment2(cx, cy, ax, ay, bx, by), point_segment2(dx, dy, ax, ay, bx, by)));
            touch = (o1 * o2 <= 0.0 && o3 * o4 <= 0.0) || d2 <= r * r;
        }
        touching[i] = touch ? (I)t : (I)(-1);
        if (touch) frame[i] = (I)(-1);
    }
    const int n = __syncthreads_count(touch);
    if (threadIdx.x == 0 && n) atomicAdd(n_touching, n);
}

// The ids of the plan tiles that hold items (in no fixed order), one atomic
// per workgroup of 256: list[0 .. *count).
__global__ void __launch_bounds__(256)
k_nonempty_tiles(const int *__restrict__ tile_off, int64_t n_tiles, int *__restrict__ list, int *__restrict__ count)
{
    __shared__ int wcnt[4];
    __shared__ int wbase[4];
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const bool ne = t < n_tiles && tile_off[t + 1] > tile_off[t];
    const uint64_t m = __ballot(ne);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wcnt[wave] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        const int total = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
        const int base = total ? atomicAdd(count, total) : 0;
        wbase[0] = base;
        wbase[1] = base + wcnt[0];
        wbase[2] = base + wcnt[0] + wcnt[1];
        wbase[3] = base + wcnt[0] + wcnt[1] + wcnt[2];
    }
    __syncthreads();
    const int below = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    if (ne) list[wbase[wave] + below] = (int)t;
}

template <typename T, int IN_OV, int OUT_OV>
static void launch_accumulate(int kernel, T *out, const SegmentPlan<T> &P, T max_val, const int32_t *frames32,
                              const int *tile_list, int64_t n_list, hipStream_t st)
{
    launch_ordered_k<T, IN_OV, 32, 16, true, OUT_OV>(kernel, out, nullptr, nullptr, P, max_val, st, frames32,
                                                     tile_list, n_list);
}

// accumulate_lines (bresenham.cpp:151-256): lines grouped into terms, each
// term reduced over its lines (in_overlap), terms reduced into frames
// (out_overlap).  Equal overlaps compose to draw_lines with idxs =
// frames[terms] on the tile path.  Different overlaps bin the lines by (term,
// tile) and run the ordered tile kernel in accumulate mode: each term tile
// is reduced in LDS in reference line order from zero, like the reference's
// term buffer, and its touched pixels are combined into frame frames[term]
// with atomics (bresenham.cpp:230-248).  Terms reach a frame in no fixed
// order, as under the reference's OpenMP loop over terms.
//
// In float images most lines of a term usually share no pixel with another line
// of it (k_term_touch).  The reduction over such a line is the line, so those
// go to the frames by the tile kernel with exact values, which is cheaper
// than a (term, tile) list each; a sum of them is rounded once instead of once
// a term.
// (term, tile) pairs of one mixed-overlap accumulate plan at most
constexpr int64_t MAX_TERM_TILES = int64_t(1) << 24;
// k_term_touch compares every pair of a term's lines (this many times the lines):
// terms of more lines leave all lines to the (term, tile) lists.
constexpr int64_t MAX_TERM_LINES = 256;
// A second plan and its launches take 70 us, and its tile kernel a workgroup per
// tile; a line alone saves some 20 ns of (term, tile) lists.  So it is made for at
// least this many such lines in at least this many tiles.  All lists / split, us, lines
// of 10 to 60 px: 1000, 4000 and 8000 lines in 1024 tiles 178 / 210, 249 / 242 and
// 336 / 264, 64 000 lines 1420 / 480; 16 000 lines in 81, 100 and 144 tiles 475 / 537,
// 485 / 493 and 504 / 440; 64 000 lines in 49 tiles 1330 / 1970.
constexpr int64_t LONE_MIN_LINES = 4096, LONE_MIN_TILES = 128;

// term of each line within the batch [t0, t1), or -1 (a line of another batch)
template <typename I>
__global__ void k_term_batch(const I *__restrict__ terms, int64_t n_lines, int64_t t0, int64_t t1,
                             I *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_lines) return;
    const int64_t t = (int64_t)terms[i];
    out[i] = (t >= t0 && t < t1) ? (I)(t - t0) : (I)(-1);
}

template <typename T, typename I>
static int accumulate_batch(T *out, const T *lines, int64_t n_lines, const I *bidx, int64_t n_terms, bool skip,
                            const int32_t *frames32, int64_t H, int64_t W, T max_val, int kernel, int in_overlap,
                            hipStream_t st);

template <typename T, typename I>
static int accumulate_lines_impl(T *out, int64_t n_frames, int64_t H, int64_t W, const T *lines, int64_t n_lines,
                                 const I *terms, const I *frames, int64_t n_terms, T max_val, int kernel,
                                 int in_overlap, int out_overlap, const cbx_draw_opts *opts, void *stream)
{
    if (in_overlap < 0 || in_overlap > 1 || out_overlap < 0 || out_overlap > 1)
        return fail(CBX_EVALUE, "Invalid in_overlap and out_overlap keywords");
    if (n_terms < 0) return fail(CBX_EVALUE, "negative size");
    if (n_lines > 0 && !terms) return fail(CBX_EVALUE, "terms must not be NULL");
    if (n_terms > 0 && !frames) return fail(CBX_EVALUE, "frames must not be NULL");
    if (n_terms >= (int64_t(1) << 31)) return fail(CBX_EVALUE, "too many terms");
    int rc = check_common(n_frames, H, W, n_lines, true, kernel, in_overlap);
    if (rc) return rc;
    if (opts && opts->kernels) return fail(CBX_EVALUE, "accumulate_lines takes one profile per call");
    hipStream_t st = (hipStream_t)stream;
    const int64_t n_chk = n_lines > n_terms ? n_lines : n_terms;
    const bool same = in_overlap == out_overlap;
    // lines alone in their pixels by frame tiles (LONE_MIN_LINES), unless a term is
    // large (surely so where the terms hold more lines on average, else counted
    // below), a tile index would not fit or max_val is not finite
    int tile = 0, seg = 0;
    resolve_opts(nullptr, n_frames, H, W, tile, seg);
    const int64_t n_tiles = n_frames * ((H + tile - 1) / tile) * ((W + tile - 1) / tile);
    bool by_tile = !same && sizeof(T) == 4 && std::isfinite(max_val) && n_lines >= LONE_MIN_LINES &&
                   n_lines <= MAX_TERM_LINES * n_terms && n_tiles >= LONE_MIN_TILES &&
                   n_tiles < (int64_t(1) << 31) / LIST_SUBS;
    DevBuf<I> comp;
    DevBuf<int32_t> frames32;
    DevBuf<int> cnt, rank;
    if (n_chk > 0) {
        DevBuf<int> bad;
        CBX_HIP(bad.alloc(3, st));
        if ((same || by_tile) && n_lines > 0) CBX_HIP(comp.alloc(n_lines, st));
        CBX_HIP(frames32.alloc(n_terms > 0 ? n_terms : 1, st));
        if (by_tile) {
            CBX_HIP(cnt.alloc(n_terms, st));
            CBX_HIP(rank.alloc(n_lines, st));
        }
        void *const zp[2] = {bad.ptr, cnt.ptr};
        const int64_t zw[2] = {3, by_tile ? n_terms : 0};
        CBX_HIP(zero_words(st, 2, zp, zw));
        k_term_frames<I><<<grid_for(n_chk, 256), 256, 0, st>>>(terms, frames, n_lines, n_terms, n_frames,
                                                                 comp.ptr, frames32.ptr, bad.ptr);
        if (by_tile)
            k_term_count<I><<<(unsigned)std::min<int64_t>(grid_for(n_lines, 256), TERM_COUNT_BLOCKS), 256, 0, st>>>(
                terms, n_lines, n_terms, (int)MAX_TERM_LINES, cnt.ptr, rank.ptr, bad.ptr + 2);
        CBX_HIP(hipGetLastError());
        const void *src[3] = {bad.ptr, bad.ptr + 1, bad.ptr + 2};
        const int nb[3] = {4, 4, 4};
        uint64_t hv[3] = {0, 0, 0};
        CBX_HIP(read_device_values(st, 3, src, nb, hv));
        if (hv[1]) return fail(CBX_EINDEX, "frames is outside of (0, n_frames)");
        if (hv[0]) return fail(CBX_EINDEX, "a term index is outside of (0, len(frames))");
        by_tile = by_tile && hv[2] == 0;
    }
    if (n_lines == 0 || n_frames * H * W == 0) return CBX_OK;
    // max/max: the term buffer starts at zero and takes std::max(buffer, v),
    // so with max_val < 0 every drawn pixel holds 0 when its term ends: the
    // draw_lines max of zero values
    if (same) return draw_lines_impl<T, I>(out, n_frames, H, W, lines, n_lines, comp.ptr,
                                           (in_overlap == 1 && max_val < T(0)) ? T(0) : max_val, kernel,
                                           in_overlap, opts, stream);

    // lines alone in their pixels: a plan of their own over the frames, drawn after the others
    SegmentPlan<T> lone;
    DevBuf<I> touching;
    int64_t n_touching = n_lines;
    if (by_tile) {
        DevBuf<int> off, order, n_dev;
        CBX_HIP(touching.alloc(n_lines, st));
        CBX_HIP(off.alloc(n_terms + 1, st));
        CBX_HIP(order.alloc(n_lines, st));
        CBX_HIP(n_dev.alloc(1, st));
        void *const zp[1] = {n_dev.ptr};
        const int64_t zw[1] = {1};
        CBX_HIP(zero_words(st, 1, zp, zw));
        CBX_HIP(exclusive_scan_total_i32(cnt.ptr, nullptr, off.ptr, n_terms, st));
        const unsigned grid = (unsigned)grid_for(n_lines, 256);
        k_term_order<I><<<grid, 256, 0, st>>>(terms, off.ptr, rank.ptr, n_lines, order.ptr);
        k_term_touch<T, I><<<grid, 256, 0, st>>>(lines, terms, off.ptr, order.ptr, n_lines, comp.ptr, touching.ptr,
                                                 n_dev.ptr);
        CBX_HIP(hipGetLastError());
        const void *src[1] = {n_dev.ptr};
        const int nb[1] = {4};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        n_touching = (int64_t)hv;
        by_tile = n_lines - n_touching >= LONE_MIN_LINES;
        if (by_tile) {
            // (checks every line: a call that fails leaves `out` untouched)
            if ((rc = build_plan_unordered<T, I>(lone, lines, comp.ptr, nullptr, kernel, n_lines, n_frames, H, W, tile,
                                                 seg, st, nullptr, false, true)))
                return rc;
        }
    }

    // The plan's frames are terms: (term, tile) lists scale with n_terms.
    // Above MAX_TERM_TILES pairs the terms go in batches, each with a plan of
    // its own (the lines of other terms skipped), in a nested workspace whose
    // memory the next batch reuses.
    const int64_t per_frame = ((H + 31) / 32) * ((W + 31) / 32);
    const int64_t batch = std::max<int64_t>(1, std::min<int64_t>(n_terms, MAX_TERM_TILES / per_frame));
    const I *const of_terms = by_tile ? touching.ptr : terms;
    DevBuf<I> bterms;
    if (batch < n_terms && n_touching > 0) CBX_HIP(bterms.alloc(n_lines, st));
    for (int64_t t0 = 0; t0 < n_terms && n_touching > 0; t0 += batch) {
        const int64_t t1 = std::min(n_terms, t0 + batch);
        Workspace inner(st);
        const I *bidx = of_terms;
        if (batch < n_terms) {
            k_term_batch<I><<<grid_for(n_lines, 256), 256, 0, st>>>(of_terms, n_lines, t0, t1, bterms.ptr);
            CBX_HIP(hipGetLastError());
            bidx = bterms.ptr;
        }
        if ((rc = accumulate_batch<T, I>(out, lines, n_lines, bidx, t1 - t0, by_tile || batch < n_terms, frames32.ptr + t0,
                                         H, W, max_val, kernel, in_overlap, st)))
            return rc;
    }
    if (by_tile && lone.n_segs > 0) {
        KernelTimer timer("accumulate_lone", st);
        cbx_draw_opts exact{};
        exact.exact_values = 1;
        // a term's buffer starts at zero: with max_val < 0 its maximum is 0
        run_tiles<T>(out, lone, kernel, out_overlap, (in_overlap == 1 && max_val < T(0)) ? T(0) : max_val, &exact, st);
        CBX_HIP(hipGetLastError());
    }
    return CBX_OK;
}

// One batch of terms of a mixed-overlap accumulate_lines: plan over the
// batch's (term, tile) pairs, tile sort, ordered render in accumulate mode.
// bidx: term of each line within the batch (negative: another batch's line).
template <typename T, typename I>
static int accumulate_batch(T *out, const T *lines, int64_t n_lines, const I *bidx, int64_t n_terms, bool skip,
                            const int32_t *frames32, int64_t H, int64_t W, T max_val, int kernel, int in_overlap,
                            hipStream_t st)
{
    int rc;
    SegmentPlan<T> P;
    if ((rc = build_plan<T, I>(P, lines, bidx, kernel, n_lines, n_terms, H, W, 32, 16, true, st, skip))) return rc;
    if (P.n_segs == 0) return CBX_OK;
    // (term, tile) pairs are mostly empty: launch over the non-empty ones only
    DevBuf<int> list, n_list;
    CBX_HIP(list.alloc(P.n_tiles, st));
    CBX_HIP(n_list.alloc(1, st));
    CBX_HIP(hipMemsetAsync(n_list.ptr, 0, sizeof(int), st));
    k_nonempty_tiles<<<grid_for(P.n_tiles, 256), 256, 0, st>>>(P.tile_off.ptr, P.n_tiles, list.ptr, n_list.ptr);
    CBX_HIP(hipGetLastError());
    int64_t nl = 0;
    {
        const void *src[1] = {n_list.ptr};
        const int nb[1] = {4};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        nl = (int64_t)(uint32_t)hv;
    }
    if (nl < 0 || nl > P.n_tiles) return fail(CBX_ERUNTIME, "non-empty tile count out of range");
    if (nl == 0) return CBX_OK;
    k_sort_tile_items<<<(unsigned)nl, 256, 0, st>>>(P.tile_off.ptr, P.items.ptr, P.flags.ptr, list.ptr);
    CBX_HIP(hipGetLastError());
    {
        KernelTimer timer("accumulate_tiles", st);
        if (in_overlap == 0) launch_accumulate<T, 0, 1>(kernel, out, P, max_val, frames32, list.ptr, nl, st);
        else launch_accumulate<T, 1, 0>(kernel, out, P, max_val, frames32, list.ptr, nl, st);
    }
    CBX_HIP(hipGetLastError());
    int fl = 0;
    {
        const void *src[1] = {P.flags.ptr};
        const int nb[1] = {4};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        fl = (int)(uint32_t)hv;
    }
    if (fl & FLAG_TILE_FULL)
        return fail(CBX_ERUNTIME, "a tile holds more than 8192 segments; accumulate_lines cannot sort it");
    return flags_to_status(fl);
}

template <typename T, int K>
static void launch_adjoint(const T *grad, const T *lines, const SegmentPlan<T> &P, const int *slot_base,
                           T max_val, double *partial, hipStream_t st)
{
    constexpr int NT = 256;
    auto run = [&](auto tile, auto seg) {
        if constexpr (sizeof(T) == 4)
            k_adjoint_fast<K, tile(), seg(), NT, 192 / seg()><<<(unsigned)P.n_tiles, NT, 0, st>>>(
                grad, lines, P.g, P.tile_off.ptr, P.pairs.ptr, P.segs.ptr, P.setup.ptr, P.lite.ptr, slot_base, max_val,
                partial, P.flags.ptr);
        else
            k_adjoint_tiles<T, K, tile(), seg(), NT, 256 / seg()><<<(unsigned)P.n_tiles, NT, 0, st>>>(
                grad, lines, P.g, P.tile_off.ptr, P.pairs.ptr, P.segs.ptr, P.setup.ptr, slot_base, max_val, partial,
                P.flags.ptr);
    };
    using std::integral_constant;
    if (P.g.tile == 64 && P.g.seg == 16) run(integral_constant<int, 64>{}, integral_constant<int, 16>{});
    else if (P.g.tile == 64) run(integral_constant<int, 64>{}, integral_constant<int, 8>{});
    else if (P.g.seg == 16) run(integral_constant<int, 32>{}, integral_constant<int, 16>{});
    else run(integral_constant<int, 32>{}, integral_constant<int, 8>{});
}

template <typename T, typename I>
static int adjoint_impl(const T *grad, int64_t n_frames, int64_t H, int64_t W, const T *lines, int64_t n_lines,
                        const I *idxs, T max_val, int kernel, T *grad_lines, const cbx_draw_opts *opts, void *stream)
{
    int rc = check_common(n_frames, H, W, n_lines, idxs != nullptr, kernel, 0);
    if (rc) return rc;
    int tile, seg;
    resolve_opts(opts, n_frames, H, W, tile, seg);
    if ((rc = check_opts(tile, seg))) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (n_lines == 0) return CBX_OK;
    CBX_HIP(hipMemsetAsync(grad_lines, 0, sizeof(T) * 5 * n_lines, st));
    if (n_frames * H * W == 0 || kernel == K_RECTANGULAR) return CBX_OK;
    SegmentPlan<T> P;
    DevBuf<int64_t> line_base;
    CBX_HIP(line_base.alloc(n_lines, st));
    if ((rc = build_plan_unordered<T, I>(P, lines, idxs, nullptr, kernel, n_lines, n_frames, H, W, tile, seg, st,
                                         line_base.ptr, true)))
        return rc;
    if (P.n_segs == 0) return CBX_OK;
    const int blk = 256;
    // each slot's first partial (tiles per slot from the binning), P.n_items
    // (< 2^31) in all
    DevBuf<int> sbase;
    CBX_HIP(sbase.alloc(P.n_segs + 1, st));
    CBX_HIP(exclusive_scan_total_i32(P.slot_tiles.ptr, nullptr, sbase.ptr, P.n_segs, st));
    // every (slot, tile) partial is written by exactly one tile
    DevBuf<double> partial;
    CBX_HIP(partial.alloc(5 * P.n_items, st));
    KernelTimer timer("adjoint_tiles", st);
    switch (kernel) {
    case K_BIWEIGHT: launch_adjoint<T, K_BIWEIGHT>(grad, lines, P, sbase.ptr, max_val, partial.ptr, st); break;
    case K_GAUSSIAN: launch_adjoint<T, K_GAUSSIAN>(grad, lines, P, sbase.ptr, max_val, partial.ptr, st); break;
    case K_PARABOLIC: launch_adjoint<T, K_PARABOLIC>(grad, lines, P, sbase.ptr, max_val, partial.ptr, st); break;
    default: launch_adjoint<T, K_TRIANGULAR>(grad, lines, P, sbase.ptr, max_val, partial.ptr, st); break;
    }
    CBX_HIP(hipGetLastError());
    k_line_grad<T><<<grid_for(n_lines * LG_LANES, blk), blk, 0, st>>>(line_base.ptr, P.setup.ptr, P.g, sbase.ptr,
                                                                      partial.ptr, n_lines, grad_lines, P.flags.ptr);
    CBX_HIP(hipGetLastError());
    int fl = 0;
    {
        const void *src[1] = {P.flags.ptr};
        const int nb[1] = {4};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        fl = (int)(uint32_t)hv;
    }
    return flags_to_status(fl);
}

} // namespace cbx

// ---------------------------------------------------------------------------
// plans: the unordered tile path sized once, then drawn without host syncs,
// allocations or memsets
// ---------------------------------------------------------------------------
struct cbx_plan {
    cbx::SegmentPlan<float> P; // capacities in P.n_segs (slots) and P.n_items
    cbx::DevBuf<unsigned long long> counters;
    cbx::DevBuf<unsigned long long> scan_state; // the tile-offset scan's look-back state
    cbx::DevBuf<int64_t> line_base;             // each line's first slot in the last draw
    // the adjoint's buffers (allocated by the plan's first adjoint; the tiles
    // per slot, P.slot_tiles, are written by every draw)
    cbx::DevBuf<int> sbase;                     // each slot's first partial
    cbx::DevBuf<double> partial;                // five partial sums per (slot, tile)
    cbx::DevBuf<unsigned long long> adj_state;  // the slot-offset scan's look-back state
    int64_t n_lines_max = 0;
    int64_t bytes = 0;
    // the last draw: line count, profile (-1: per-line profiles)
    int64_t last_lines = -1;
    int last_kernel = -1;
    cbx_draw_opts opts{};
};

namespace cbx {

static int plan_create(cbx_plan **out_plan, int64_t n_frames, int64_t H, int64_t W, const float *lines,
                       int64_t n_lines, const int32_t *idxs, const uint8_t *kernels, int kernel,
                       const cbx_draw_opts *opts, double headroom, hipStream_t st)
{
    if (!out_plan) return fail(CBX_EVALUE, "plan must not be NULL");
    *out_plan = nullptr;
    int rc = check_common(n_frames, H, W, n_lines, idxs != nullptr, kernel, 0);
    if (rc) return rc;
    if (!(headroom >= 1.0) || headroom > 64.0) return fail(CBX_EVALUE, "headroom must be in [1, 64]");
    if (n_lines <= 0 || n_frames * H * W == 0) return fail(CBX_EVALUE, "a plan needs lines and a non-empty frame");
    int tile, seg;
    resolve_opts(opts, n_frames, H, W, tile, seg);
    if ((rc = check_opts(tile, seg))) return rc;
    if (opts && !(opts->threads == 0 || opts->threads == 64 || opts->threads == 128 || opts->threads == 256))
        return fail(CBX_EVALUE, "threads must be 64, 128 or 256");
    if (opts && opts->deterministic) return fail(CBX_EVALUE, "plans draw with the tile path (deterministic = 0)");
    // sizing pass on the given lines (intermediates from the workspace cache)
    int64_t slots = 0, items = 0;
    {
        Workspace ws(st);
        SegmentPlan<float> S;
        if ((rc = build_plan_unordered<float, int32_t>(S, lines, idxs, kernels, kernel, n_lines, n_frames, H, W, tile,
                                                        seg, st)))
            return rc;
        slots = S.n_segs;
        items = S.n_items;
    }
    const int64_t slot_cap = std::max<int64_t>((int64_t)std::ceil((double)slots * headroom), slots + 1024);
    const int64_t item_cap = std::max<int64_t>((int64_t)std::ceil((double)items * headroom), items + 1024);
    if (slot_cap >= (int64_t(1) << 31) || item_cap >= (int64_t(1) << 31))
        return fail(CBX_EVALUE, "plan capacity exceeds 2^31 entries");
    cbx_plan *pl = new cbx_plan();
    SegmentPlan<float> &P = pl->P;
    Geometry &g = P.g;
    g.n_frames = n_frames;
    g.H = (int32_t)H;
    g.W = (int32_t)W;
    set_tiles(g, tile, seg);
    P.n_lines = n_lines;
    P.n_tiles = n_frames * g.ntx * g.nty;
    const int64_t n_lists = P.n_tiles * LIST_SUBS;
    P.n_segs = slot_cap;
    P.n_items = item_cap;
    pl->n_lines_max = n_lines;
    if (opts) pl->opts = *opts;
    pl->opts.kernels = nullptr;
    pl->opts.tile = tile;
    pl->opts.seg = seg;
    hipError_t e = hipSuccess;
    auto take = [&](hipError_t r) {
        if (e == hipSuccess) e = r;
    };
    // owned allocations (no workspace is open here)
    take(P.setup.alloc(n_lines, st));
    take(P.lite.alloc(n_lines, st));
    take(P.flags.alloc(1, st));
    take(P.segs.alloc(slot_cap, st));
    take(P.slot_tiles.alloc(slot_cap, st));
    take(P.tile_cnt.alloc(n_lists, st));
    take(P.tile_off.alloc(n_lists + 1, st));
    take(P.tile_cur.alloc(n_lists, st));
    take(P.pairs.alloc(item_cap, st));
    take(pl->counters.alloc(2, st));
    take(pl->line_base.alloc(n_lines, st));
    const size_t scan_words = scan_state_words(n_lists + 1);
    take(pl->scan_state.alloc(scan_words, st));
    if (e == hipSuccess) e = clear_scan_state(pl->scan_state.ptr, scan_words, st);
    if (e != hipSuccess) {
        delete pl;
        return fail(CBX_ERUNTIME, std::string("plan allocation: ") + hipGetErrorString(e));
    }
    pl->bytes = (int64_t)((sizeof(LineSetup<float>) + sizeof(LineLite) + sizeof(int64_t)) * n_lines +
                          (sizeof(Segment<float>) + sizeof(int)) * slot_cap +
                          sizeof(int2) * item_cap + 3 * sizeof(int) * n_lists + sizeof(int) +
                          sizeof(unsigned long long) * scan_words);
    *out_plan = pl;
    return CBX_OK;
}

static int plan_draw(cbx_plan *pl, float *out, const float *lines, int64_t n_lines, const int32_t *idxs,
                     const uint8_t *kernels, float max_val, int kernel, int overlap, hipStream_t st)
{
    if (!pl) return fail(CBX_EVALUE, "plan must not be NULL");
    SegmentPlan<float> &P = pl->P;
    int rc = check_common(P.g.n_frames, P.g.H, P.g.W, n_lines, idxs != nullptr, kernel, overlap);
    if (rc) return rc;
    if (n_lines > pl->n_lines_max) return fail(CBX_EVALUE, "more lines than the plan was created for");
    if (n_lines == 0) return CBX_OK;
    const int blk = 256;
    const Geometry &g = P.g;
    const int64_t n_lists = P.n_tiles * LIST_SUBS;
    const int64_t reset_n = std::max<int64_t>(n_lists, (int64_t)pl->scan_state.n);
    k_plan_reset<<<grid_for(reset_n, blk), blk, 0, st>>>(n_lists, pl->counters.ptr, P.flags.ptr, P.tile_cnt.ptr,
                                                         P.tile_cur.ptr, pl->scan_state.ptr,
                                                         (int64_t)pl->scan_state.n);
    k_setup_lines<float, int32_t><<<grid_for(n_lines, blk), blk, 0, st>>>(lines, idxs, kernels, kernel, n_lines, g,
                                                                         P.setup.ptr, P.lite.ptr, pl->counters.ptr, P.flags.ptr);
    k_walk_lines<float><<<grid_for(n_lines, blk), blk, 0, st>>>(n_lines, g, P.setup.ptr, P.segs.ptr, P.n_segs,
                                                                pl->counters.ptr, P.tile_cnt.ptr, P.flags.ptr,
                                                                pl->line_base.ptr);
    // the plan's own scan state (cleared by k_plan_reset above)
    CBX_HIP(scan_i32_with_state(P.tile_cnt.ptr, nullptr, P.tile_off.ptr, n_lists, n_lists + 1, pl->scan_state.ptr,
                                st));
    k_bin_slots<float><<<grid_for(P.n_segs, blk), blk, 0, st>>>(P.n_segs, g, P.setup.ptr, P.segs.ptr,
                                                                P.tile_off.ptr, P.tile_cur.ptr, P.pairs.ptr,
                                                                pl->counters.ptr, P.n_tiles, P.n_items, P.flags.ptr,
                                                                P.slot_tiles.ptr);
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(st, &cap);
    if (cap == hipStreamCaptureStatusNone) {
        KernelTimer timer("draw_tiles", st);
        run_tiles<float>(out, P, kernels ? K_MIXED : kernel, overlap, max_val, &pl->opts, st);
    } else {
        run_tiles<float>(out, P, kernels ? K_MIXED : kernel, overlap, max_val, &pl->opts, st);
    }
    CBX_HIP(hipGetLastError());
    pl->last_lines = n_lines;
    pl->last_kernel = kernels ? -1 : kernel;
    return CBX_OK;
}

// The adjoint of the plan's last draw, on its segments and tile lists (no
// second walk): the same kernels as cbx_draw_lines_adjoint_f32, with no host
// synchronisation; errors of the draw leave grad_lines zero and are reported
// by plan_check.  The first call allocates the adjoint's buffers.
static int plan_adjoint(cbx_plan *pl, const float *grad, const float *lines, int64_t n_lines, const int32_t *idxs,
                        float max_val, int kernel, float *grad_lines, hipStream_t st)
{
    if (!pl) return fail(CBX_EVALUE, "plan must not be NULL");
    SegmentPlan<float> &P = pl->P;
    int rc = check_common(P.g.n_frames, P.g.H, P.g.W, n_lines, idxs != nullptr, kernel, 0);
    if (rc) return rc;
    if (n_lines == 0) return CBX_OK;
    if (pl->last_kernel < 0 && pl->last_lines >= 0)
        return fail(CBX_EVALUE, "the plan's last draw used per-line profiles: no adjoint");
    if (n_lines != pl->last_lines || kernel != pl->last_kernel)
        return fail(CBX_EVALUE, "the adjoint needs the line count and profile of the plan's last draw");
    if (!pl->partial.ptr) {
        hipError_t e = pl->sbase.alloc(P.n_segs + 1, st);
        if (e == hipSuccess) e = pl->partial.alloc(5 * P.n_items, st);
        if (e == hipSuccess) e = pl->adj_state.alloc(scan_state_words(P.n_segs + 1), st);
        if (e != hipSuccess) {
            pl->partial.release();
            return fail(CBX_ERUNTIME, std::string("plan adjoint allocation: ") + hipGetErrorString(e));
        }
        pl->bytes += (int64_t)(sizeof(int) * (P.n_segs + 1) + sizeof(double) * 5 * P.n_items +
                               sizeof(unsigned long long) * pl->adj_state.n);
    }
    {
        // the gradient and the scan's state, cleared by one kernel
        void *const zp[2] = {grad_lines, pl->adj_state.ptr};
        const int64_t zw[2] = {5 * n_lines, 2 * (int64_t)pl->adj_state.n};
        CBX_HIP(zero_words(st, 2, zp, zw));
    }
    if (kernel == K_RECTANGULAR) return CBX_OK;   // a flat profile: zero gradient
    const int blk = 256;
    CBX_HIP(scan_i32_with_state(P.slot_tiles.ptr, nullptr, pl->sbase.ptr, P.n_segs, P.n_segs + 1, pl->adj_state.ptr,
                                st));
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(st, &cap);
    {
        KernelTimer timer(cap == hipStreamCaptureStatusNone ? "adjoint_tiles" : nullptr, st);
        switch (kernel) {
        case K_BIWEIGHT: launch_adjoint<float, K_BIWEIGHT>(grad, lines, P, pl->sbase.ptr, max_val, pl->partial.ptr, st); break;
        case K_GAUSSIAN: launch_adjoint<float, K_GAUSSIAN>(grad, lines, P, pl->sbase.ptr, max_val, pl->partial.ptr, st); break;
        case K_PARABOLIC: launch_adjoint<float, K_PARABOLIC>(grad, lines, P, pl->sbase.ptr, max_val, pl->partial.ptr, st); break;
        default: launch_adjoint<float, K_TRIANGULAR>(grad, lines, P, pl->sbase.ptr, max_val, pl->partial.ptr, st); break;
        }
    }
    k_line_grad<float><<<grid_for(n_lines * LG_LANES, blk), blk, 0, st>>>(
        pl->line_base.ptr, P.setup.ptr, P.g, pl->sbase.ptr, pl->partial.ptr, n_lines, grad_lines, P.flags.ptr);
    CBX_HIP(hipGetLastError());
    return CBX_OK;
}

static int plan_check(cbx_plan *pl, hipStream_t st)
{
    if (!pl) return fail(CBX_EVALUE, "plan must not be NULL");
    int fl = 0;
    {
        const void *src[1] = {pl->P.flags.ptr};
        const int nb[1] = {4};
        uint64_t hv = 0;
        CBX_HIP(read_device_values(st, 1, src, nb, &hv));
        fl = (int)(uint32_t)hv;
    }
    return flags_to_status(fl);
}

} // namespace cbx

extern "C" {

int cbx_plan_create_f32(cbx_plan **plan, int64_t n_frames, int64_t height, int64_t width, const float *lines,
                        int64_t n_lines, const int32_t *idxs, const uint8_t *kernels, int kernel,
                        const cbx_draw_opts *opts, double headroom, void *stream)
{
    return cbx::plan_create(plan, n_frames, height, width, lines, n_lines, idxs, kernels, kernel, opts, headroom,
                            (hipStream_t)stream);
}

int cbx_plan_draw_f32(cbx_plan *plan, float *out, const float *lines, int64_t n_lines, const int32_t *idxs,
                      const uint8_t *kernels, float max_val, int kernel, int overlap, void *stream)
{
    return cbx::plan_draw(plan, out, lines, n_lines, idxs, kernels, max_val, kernel, overlap, (hipStream_t)stream);
}

int cbx_plan_adjoint_f32(cbx_plan *plan, const float *grad_out, const float *lines, int64_t n_lines,
                         const int32_t *idxs, float max_val, int kernel, float *grad_lines, void *stream)
{
    return cbx::plan_adjoint(plan, grad_out, lines, n_lines, idxs, max_val, kernel, grad_lines, (hipStream_t)stream);
}

int cbx_plan_check(cbx_plan *plan, void *stream) { return cbx::plan_check(plan, (hipStream_t)stream); }

int64_t cbx_plan_bytes(const cbx_plan *plan) { return plan ? plan->bytes : 0; }

void cbx_plan_destroy(cbx_plan *plan)
{
    if (!plan) return;
    (void)hipDeviceSynchronize();
    delete plan;
}

} // extern "C"

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int cbx_draw_lines_f32(float *out, int64_t n_frames, int64_t height, int64_t width, const float *lines,
                       int64_t n_lines, const int32_t *idxs, float max_val, int kernel, int overlap,
                       const cbx_draw_opts *opts, void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::draw_lines_impl<float, int32_t>(out, n_frames, height, width, lines, n_lines, idxs, max_val, kernel,
                                                overlap, opts, stream);
}

int cbx_draw_lines_f64(double *out, int64_t n_frames, int64_t height, int64_t width, const double *lines,
                       int64_t n_lines, const int64_t *idxs, double max_val, int kernel, int overlap,
                       const cbx_draw_opts *opts, void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::draw_lines_impl<double, int64_t>(out, n_frames, height, width, lines, n_lines, idxs, max_val, kernel,
                                                 overlap, opts, stream);
}

int cbx_draw_pixels_f32(int64_t n_frames, int64_t height, int64_t width, const float *lines, int64_t n_lines,
                        const int32_t *idxs, float max_val, int kernel, int overlap, int merge, int32_t *frame,
                        int32_t *y, int32_t *x, float *value, int32_t *line, int64_t capacity, int64_t *count,
                        void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::draw_pixels_impl<float, int32_t>(n_frames, height, width, lines, n_lines, idxs, max_val, kernel,
                                                 overlap, merge, frame, y, x, value, line, capacity, count, stream);
}

int cbx_draw_pixels_f64(int64_t n_frames, int64_t height, int64_t width, const double *lines, int64_t n_lines,
                        const int64_t *idxs, double max_val, int kernel, int overlap, int merge, int32_t *frame,
                        int32_t *y, int32_t *x, double *value, int32_t *line, int64_t capacity, int64_t *count,
                        void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::draw_pixels_impl<double, int64_t>(n_frames, height, width, lines, n_lines, idxs, max_val, kernel,
                                                  overlap, merge, frame, y, x, value, line, capacity, count, stream);
}

int cbx_accumulate_lines_f32(float *out, int64_t n_frames, int64_t height, int64_t width, const float *lines,
                             int64_t n_lines, const int32_t *terms, const int32_t *frames, int64_t n_terms,
                             float max_val, int kernel, int in_overlap, int out_overlap, const cbx_draw_opts *opts,
                             void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::accumulate_lines_impl<float, int32_t>(out, n_frames, height, width, lines, n_lines, terms, frames,
                                                      n_terms, max_val, kernel, in_overlap, out_overlap, opts,
                                                      stream);
}

int cbx_accumulate_lines_f64(double *out, int64_t n_frames, int64_t height, int64_t width, const double *lines,
                             int64_t n_lines, const int64_t *terms, const int64_t *frames, int64_t n_terms,
                             double max_val, int kernel, int in_overlap, int out_overlap, const cbx_draw_opts *opts,
                             void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::accumulate_lines_impl<double, int64_t>(out, n_frames, height, width, lines, n_lines, terms, frames,
                                                       n_terms, max_val, kernel, in_overlap, out_overlap, opts,
                                                       stream);
}

int cbx_draw_lines_adjoint_f32(const float *grad_out, int64_t n_frames, int64_t height, int64_t width,
                               const float *lines, int64_t n_lines, const int32_t *idxs, float max_val, int kernel,
                               float *grad_lines, const cbx_draw_opts *opts, void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::adjoint_impl<float, int32_t>(grad_out, n_frames, height, width, lines, n_lines, idxs, max_val, kernel,
                                             grad_lines, opts, stream);
}

int cbx_draw_lines_adjoint_f64(const double *grad_out, int64_t n_frames, int64_t height, int64_t width,
                               const double *lines, int64_t n_lines, const int64_t *idxs, double max_val,
                               int kernel, double *grad_lines, const cbx_draw_opts *opts, void *stream)
{
    cbx::Workspace ws((hipStream_t)stream);
    return cbx::adjoint_impl<double, int64_t>(grad_out, n_frames, height, width, lines, n_lines, idxs, max_val,
                                              kernel, grad_lines, opts, stream);
}

} // extern "C"
