// Types of the 2D draw pipeline shared by its translation units: segments,
// line records, the plan of a draw, the walk replay and the column fills.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "cbx_core.hpp"
#include "cbx_host.hpp"

namespace cbx {

template <typename T>
struct Segment {
    int32_t line;
    int32_t c[2];   // walk position at the segment's first column
    int32_t ncols;  // emitted long-axis columns, consecutive from c[axis] in the walk direction
    T Te, Ne;       // walk errors at that position
    int32_t lo, hi; // short-axis pixel range the fills can reach, clipped to the frame
};

// What the float tile kernel needs of a line (32 bytes, two 16-byte loads; the
// whole LineSetup is read only for exact errors next to the threshold and for
// the lines that are not FR_SAFE).
struct alignas(16) LineLite {
    float t[2];       // tangent (the normal components are t[1], -t[0])
    float LL, ea;     // as in LineSetup
    float nlim;       // band limit
    float cap;        // a column with cap < Te < LL - cap has no tangential overshoot at any of its pixels
    int32_t meta;     // FR_* bits, profile id in bits 8-15
};
constexpr int FR_AXIS = 1, FR_SA = 2, FR_SB = 4, FR_SAFE = 8;

struct Geometry {
    int64_t n_frames;
    int32_t H, W;
    int32_t tile, seg;
    int32_t tile_log, seg_log;
    int32_t ntx, nty;
    uint32_t m_frame = 0, m_ntx = 0;   // tile_coords: 2^32 / (tiles per frame), 2^32 / ntx, rounded down
    int32_t skip_neg = 0;   // 1: a line with a negative frame draws nothing (accumulate_lines: another plan's lines)
};

// The unordered plan's item list of tile t is split into LIST_SUBS sub-lists by
// what an item costs (list_class); the sub-lists are contiguous: tile t's items
// are [tile_off[t * LIST_SUBS], tile_off[(t + 1) * LIST_SUBS]).
constexpr int LIST_SUBS = 8;

// n / d (remainder in r) from m = floor(2^32 / d) (2^32 - 1 for d = 1): the product
// is at most one too small.  Scalar instructions for a uniform n, where the
// compiler's integer division takes about 20 vector ones.
__host__ __device__ __forceinline__ uint32_t div_magic(uint32_t d)
{
    return d <= 1 ? 0xffffffffu : (uint32_t)((uint64_t(1) << 32) / d);
}
__device__ __forceinline__ int div_by(int n, int d, uint32_t m, int &r)
{
    int q = (int)__umulhi((uint32_t)n, m);
    r = n - q * d;
    if (r >= d) {
        q++;
        r -= d;
    }
    return q;
}

// frame and tile column / row of a tile index
__device__ __forceinline__ void tile_coords(const Geometry &g, int tile, int64_t &f, int &tx, int &ty)
{
    int r;
    f = div_by(tile, g.ntx * g.nty, g.m_frame, r);
    ty = div_by(r, g.ntx, g.m_ntx, tx);
}

inline void set_tiles(Geometry &g, int tile, int seg)
{
    g.tile = tile;
    g.seg = seg;
    g.tile_log = (tile == 64) ? 6 : 5;
    g.seg_log = (seg == 16) ? 4 : 3;
    g.ntx = (int32_t)((g.W + tile - 1) / tile);
    g.nty = (int32_t)((g.H + tile - 1) / tile);
    g.m_frame = div_magic((uint32_t)((int64_t)g.ntx * g.nty));
    g.m_ntx = div_magic((uint32_t)g.ntx);
}

// Sub-list of a line's items: with per-line profiles the profile, else the height
// of its band of pixels in half octaves, so that the lanes of a wave, whose items
// are neighbours in a list, run the same loop about equally long.  (962 000
// lines of mixed profiles: tile kernel 2782 -> 2684 us, by height 2747; 160 000
// lines of widths 2 to 6: 349 -> 335, their gradient 620 -> 597; quarter octaves in
// 16 sub-lists gave no more.)
template <typename T>
__device__ __forceinline__ int list_class(const LineSetup<T> &L, bool mixed)
{
    if (mixed) return L.kid & (LIST_SUBS - 1);
    const float h = (float)L.w * (float)L.len / (float)m_abs((L.axis == 0) ? L.t[0] : L.t[1]);
    return (int)__builtin_fminf(__builtin_fmaxf(2.0f * __builtin_log2f(h), 0.0f), (float)(LIST_SUBS - 1));
}

// ---------------------------------------------------------------------------
// shared pieces of the tile kernels
// ---------------------------------------------------------------------------
template <typename T>
struct ColRec {
    int32_t s; // short-axis centre, INT_MIN when the column is not emitted
    T Te, Ne;
};

struct ItemHdr {
    int32_t seg;
    int32_t line;
};

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Phase 1: replay a segment's walk from its checkpoint and record, for each
// of its columns, the centre and errors at which the reference emits it, in
// the column slots i * SEG + k of item i of rr.
template <typename T, int SEG>
__device__ __forceinline__ void walk_columns(const LineSetup<T> &L, const Segment<T> &sg, ColRec<T> *rr, int i,
                                             int *flags)
{
    for (int k = 0; k < SEG; k++) rr[i * SEG + k].s = INT_MIN;
    const int a = L.axis, b = 1 - a, sa = pick(L.st, a);
    WalkState<T> s;
    s.c[0] = sg.c[0];
    s.c[1] = sg.c[1];
    s.Te = sg.Te;
    s.Ne = sg.Ne;
    const int c0 = pick(s.c, a);
    int it = 0;
    for (; it < 4 * SEG + 16; it++) {
        if (walk_done(L, s)) break;
        const int k = (pick(s.c, a) - c0) * sa;
        if (k >= sg.ncols) break;
        bool nx, ny;
        walk_next(L, s.Ne, nx, ny);
        if ((a == 0) ? nx : ny) {
            ColRec<T> &r = rr[i * SEG + k];
            r.s = pick(s.c, b);
            r.Te = s.Te;
            r.Ne = s.Ne;
        }
        walk_step(L, s, nx, ny);
    }
    if (it == 4 * SEG + 16) atomicOr(flags, FLAG_STUCK);
}

// Phase 2: the orthogonal fills of one emitted column (bresenham.hpp:364-380),
// restricted to the short-axis window [s_lo, s_hi); emit(s, err) is called
// for every pixel of the window the reference would hand to draw_pixel.
template <typename T, typename Emit>
__device__ __forceinline__ void fill_column(const LineSetup<T> &L, const ColRec<T> &cr, int s_lo, int s_hi,
                                            Emit &&emit)
{
    const int b = 1 - L.axis;
    if (cr.s >= s_lo && cr.s < s_hi) emit(cr.s, cr.Te, cr.Ne);
    const T tb = pick(L.t, b), nb = pick(L.nv, b);
    const int sb = pick(L.st, b);
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const int dir = half ? -sb : sb;
        const T dT = (dir > 0) ? tb : -tb, dN = (dir > 0) ? nb : -nb;
        int s = cr.s;
        T Te = cr.Te, Ne = cr.Ne;
        for (;;) {
            s += dir;
            Te += dT;
            Ne += dN;
            if (!(nsq_of(L, Ne) < L.w2)) break;
            if (s >= s_lo && s < s_hi) emit(s, Te, Ne);
            else if ((dir > 0) ? (s >= s_hi) : (s < s_lo)) break;
        }
    }
}

// A wave's column records in LDS: errors and centre (relative to the item's first
// position along the short axis, in the low half of a word) of column u = slot.
template <int NREC>
struct WaveCols {
    float N[NREC], T[NREC];
    int32_t S[NREC];
    __device__ __forceinline__ int centre(int u) const { return (int)*reinterpret_cast<const int16_t *>(&S[u]); }
};

// One lane replays one segment's walk and records its ncols columns from slot
// `first` on; false if it does not end within the step budget.  A step per turn
// of the loop; its column is recorded over and over until the step that leaves
// it.  The loop is most of what a narrow line costs the tile kernels, so the
// slot (as a byte offset) and the short-axis position share one register whose
// increments along x and y are known before: 20 vector instructions a step, 31
// with separate ones (962 000 lines in 16-column segments: tile kernel 2684 ->
// 2540 us).
template <int SEG, int NREC>
__device__ __forceinline__ bool replay_columns(WaveCols<NREC> &w, const LineLite &L, const Segment<float> &sg,
                                               int first, int ncols)
{
    static_assert(NREC * 4 <= 0xffff && 4 * SEG + 16 < 0x7fff, "two 16-bit halves");
    const bool ax = L.meta & FR_AXIS, pa = L.meta & FR_SA, pb = L.meta & FR_SB;
    const bool p0 = ax ? pb : pa, p1 = ax ? pa : pb;   // steps along x and y
    const float t0 = L.t[0], t1 = L.t[1];
    const float dx = p0 ? t1 : -t1, dy = p1 ? -t0 : t0;
    const float ux = p0 ? t0 : -t0, uy = p1 ? t1 : -t1;
    const uint32_t side = pb ? 0x10000u : 0xffff0000u;
    const uint32_t ix = ax ? side : 4u, iy = ax ? 4u : side;
    typedef __attribute__((address_space(3))) char lds_char;
    typedef __attribute__((address_space(3))) float lds_float;
    typedef __attribute__((address_space(3))) int16_t lds_short;
    const uint32_t base = (uint32_t)(uintptr_t)(lds_char *)reinterpret_cast<char *>(&w);   // (LDS addresses: 16 bits)
    float Te = sg.Te, Ne = sg.Ne;
    uint32_t at = base + (uint32_t)first * 4u, o = at;
    const uint32_t stop = o + (uint32_t)ncols * 4u;
    int it = 0;
    if (o < stop)
        do {
            *(lds_float *)(uintptr_t)o = Ne;
            *(lds_float *)(uintptr_t)(o + NREC * 4) = Te;
            *(lds_short *)(uintptr_t)(o + NREC * 8) = (int16_t)(at >> 16);
            const float ex = Ne + dx, ey = Ne + dy, exy = ex + dy;
            const bool yb = __builtin_fabsf(ey) < __builtin_fabsf(ex);
            const float m = yb ? ey : ex;
            const bool both = __builtin_fabsf(exy) < __builtin_fabsf(m);
            const bool y_only = yb & !both, y = yb | both;
            Te += y_only ? 0.0f : ux;
            Te += y ? uy : 0.0f;
            Ne = both ? exy : m;
            at += y_only ? 0u : ix;
            at += y ? iy : 0u;
            o = at & 0xffffu;
            it++;
        } while ((o < stop) & (it < 4 * SEG + 16));
    asm("" : "+v"(o));   // (compare once, here: not in every turn as part of the loop's masks)
    return o >= stop;
}

typedef float v4f __attribute__((ext_vector_type(4)));

template <typename T>
struct SegmentPlan {
    Geometry g;
    int64_t n_lines = 0;
    int64_t n_segs = 0;
    int64_t n_items = 0;
    int64_t n_tiles = 0;
    DevBuf<LineSetup<T>> setup;
    DevBuf<LineLite> lite;   // unordered float plan
    DevBuf<int> seg_cnt, seg_off, tile_cnt, tile_off, tile_cur, items, flags;
    DevBuf<int2> pairs; // unordered plan: per-tile (segment, line) lists
    DevBuf<int> slot_tiles; // unordered plan, when asked for: tiles per segment slot (the adjoint's)
    DevBuf<Segment<T>> segs;
};

// Tiles of a few items each, and more of them than run at a time (four workgroups on each
// of 256 CUs): the tile kernel that holds less of a tile (FEW).  us without / with it for
// 64 frames of 1024^2 with 2, 8, 12, 16 and 24 items in a tile: sums 123 / 109, 164 / 159,
// 175 / 173, 182 / 186, 199 / 212; maxima 107 / 104, 146 / 141, 157 / 150, 167 / 160, 188 / 180.
template <typename T>
inline bool few_items(const SegmentPlan<T> &P)
{
    return P.n_tiles > 1024 && P.n_items < 12 * P.n_tiles;
}

// The tile kernel of one profile (CBX_PROFILE of cbx_tiles.hip; K_MIXED: per-line
// profiles) over a built unordered plan.
template <typename T, int K>
void run_tiles_profile(T *out, const SegmentPlan<T> &P, T max_val, int overlap, const cbx_draw_opts *opts,
                       hipStream_t st);

} // namespace cbx
