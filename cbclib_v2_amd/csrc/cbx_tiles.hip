// Tile kernels of draw_lines: the images of a built unordered plan (segments
// and per-tile item lists).  Compiled once per profile: CBX_PROFILE is one of
// cbx_core.hpp's Profile values or K_MIXED (5, each line with its own).
#include <hip/hip_runtime.h>

#include <climits>
#include <cmath>

#include "cbx_draw.hpp"

#ifndef CBX_PROFILE
#error "CBX_PROFILE: the profile this translation unit draws"
#endif

namespace cbx {

// LDS accumulator of the tile kernel, by accumulation mode OV:
//   0  sums in double (on gfx950 ds_add_f64 sustains ~20x the lane rate of
//      ds_add_f32; the tile is rounded to the image type once, at the flush)
//   1  max overlap, as order-preserving unsigned codes (ds_max)
//   2  float sums in 32-bit fixed point (ds_add_u32, the fastest LDS atomic,
//      at half the LDS of double; see k_tiles)
template <typename T, int OV>
struct AccType {
    using type = double;
};
template <>
struct AccType<float, 1> {
    using type = uint32_t;
};
template <>
struct AccType<double, 1> {
    using type = unsigned long long;
};
template <>
struct AccType<float, 2> {
    using type = uint32_t;
};

// Adds one pixel value to the LDS tile.  For OV = 2, v is the profile value
// already scaled by the round's 2^F; exact zeros only mark the pixel touched.
// POS: v is known to be positive (and, for OV = 2, at least 1).
template <int OV, bool POS = false, typename Acc, typename V>
__device__ __forceinline__ void tile_put(Acc *img, uint32_t *zb, int idx, V v)
{
    if constexpr (OV == 0) {
        atomicAdd(&img[idx], (Acc)v);
    } else if constexpr (OV == 1) {
        if (v == v) atomicMax(&img[idx], ord_enc(v));
    } else if constexpr (POS) {
        atomicAdd(&img[idx], __float2uint_rn((float)v));
    } else {
        if (v > 0.0f) atomicAdd(&img[idx], max(1u, __float2uint_rn((float)v)));
        else atomicOr(&zb[idx >> 5], 1u << (idx & 31));
    }
}

// ---------------------------------------------------------------------------
// 4. tile kernel (image mode)
// ---------------------------------------------------------------------------
// Per-item record in LDS, written by the phase-1 thread that replays the
// item's walk (it holds the line's setup in registers) and read by the
// phase-2 threads of its columns: the item's line and first long-axis
// coordinate, and for float lines the fast path's constants, so the fills
// need no global load (the exact error near the threshold reads the setup).
struct alignas(16) FillRec {
    float LL, ea, nlim;
    float tb, nb;     // tangent and normal components along the short axis b
    int32_t c0;       // long-axis coordinate of the item's first column (k_tiles_fast: short-axis position there)
    int32_t line;
    int32_t meta;     // FR_* bits, profile id in bits 8-15 (k_tiles_fast: columns from bit 16)
};

template <typename T>
__device__ __forceinline__ FillRec fill_rec(const LineSetup<T> &L, int c0, int line)
{
    FillRec r;
    const int a = L.axis, b = 1 - a;
    r.c0 = c0;
    r.line = line;
    r.meta = a | (pick(L.st, a) > 0 ? FR_SA : 0) | (pick(L.st, b) > 0 ? FR_SB : 0) |
             (sizeof(T) == 4 && L.safe ? FR_SAFE : 0) | ((int)L.kid << 8);
    r.LL = (float)L.LL;
    r.ea = L.ea;
    r.nlim = L.nlim;
    r.tb = (float)pick(L.t, b);
    r.nb = (float)pick(L.nv, b);
    return r;
}

// The fills of one column half for the float fast path (lines with L.safe):
// the band test |Ne| < nlim, the one-product error estimate (err_fast), the
// profile's constant folded into the column's value scale and the tile window
// turned into a skip count and a trip count, with the LDS index stepped per
// pixel.  The errors advance by the same FP32 additions as the reference's
// loop.  Lg is the line's setup in global memory, read only for exact errors
// near the threshold.  vscale is max_val (OV 0, 1) or the fixed-point scale
// 2^F (OV 2: F >= 20, so positive profiles give values of at least 1).
template <int K, int OV, typename Acc>
__device__ __forceinline__ void fill_half_fast(Acc *img, uint32_t *zb, const FillRec &R,
                                               const LineSetup<float> &Lg, int cs, float Te, float Ne, int half,
                                               int cbase, int sstride, int s_lo, int s_hi, float vscale)
{
    constexpr bool POS = (OV == 2) && fast_positive<K>();
    const float LL = R.LL, ea = R.ea, nlim = R.nlim;
    const int kid = (R.meta >> 8) & 0xff;
    const int sb = (R.meta & FR_SB) ? 1 : -1;
    const int dir = half ? -sb : sb;
    const float dT = (dir > 0) ? R.tb : -R.tb, dN = (dir > 0) ? R.nb : -R.nb;
    const float c = fast_scale<K>(kid, vscale);
    auto put = [&](int idx, float T, float N) {
        const float e = err_fast(Lg, LL, ea, T, N);
        if (e <= 1.0f) tile_put<OV, POS>(img, zb, idx, fast_value<K>(kid, e, c));
    };
    wait_lds_loads();
    if (half == 0 && cs >= s_lo && cs < s_hi) put(cbase + (cs - s_lo) * sstride, Te, Ne);
    // steps to the last in-window pixel in the direction of travel, and the
    // first step that lands inside the window
    const int nsteps = (dir > 0) ? (s_hi - 1 - cs) : (cs - s_lo);
    if (nsteps < 1) return;
    const int jin = max(1, (dir > 0) ? (s_lo - cs) : (cs - s_hi + 1));
    for (int j = 1; j < jin; j++) {
        Te += dT;
        Ne += dN;
        if (!(__builtin_fabsf(Ne) < nlim)) return;
    }
    const int step = dir * sstride;
    int idx = cbase + (cs + jin * dir - s_lo) * sstride;
    for (int j = jin; j <= nsteps; j++, idx += step) {
        Te += dT;
        Ne += dN;
        if (!(__builtin_fabsf(Ne) < nlim)) return;
        put(idx, Te, Ne);
    }
}

// Value a fixed-point tile pixel adds to the image: acc * max_val * 2^-F, or
// max_val * 0 (the sign rules of adding exact zeros) if only zeros touched
// it.  has = false: the pixel was not touched.
__device__ __forceinline__ double fix_value(uint32_t acc, const uint32_t *zb, int i, double scale, float max_val,
                                            bool &has)
{
    has = acc != 0u || ((zb[i >> 5] >> (i & 31)) & 1u);
    return acc ? (double)acc * scale : (double)(max_val * 0.0f);
}

// fix_value for a pixel already in a register, in float: o + (acc 2^-F)
// max_val (or + zero, the value of exact zeros, when only zeros touched it:
// zbit set), or o untouched.  acc 2^-F is exact (p2 = 2^-F); the rounding of
// acc to 24 bits and of the two operations stays below 2e-7 of the pixel's
// value, far inside the fixed-point terms' own error (<= 2^-F max_val each).
__device__ __forceinline__ float fold_fix(float o, uint32_t acc, uint32_t zbit, float p2, float max_val, float zero)
{
    const float add = acc ? ((float)acc * p2) * max_val : zero;
    return (acc | zbit) ? o + add : o;
}

// Fixed-point sums (OV = 2): an item (one segment in one tile) adds at most
// one value per pixel, so a round of n items adds at most n values of at most
// 2^F with F = clz(n): the sum stays below 2^32.  Each value p > 0 adds
// max(1, rn(p 2^F)) (absolute error <= 2^-(F+1) max_val per term, at most 2^-F
// where a touched pixel is kept non-zero); exact zeros set a bit in zb.  Tiles
// of more than FIX_ROUND items take several rounds, folded into the running
// pixel values: F >= 22, so that eight faint terms stay within 1e-6 max_val.
constexpr int FIX_ROUND = 1023;

// Tile kernel of the double images, of exact values and of non-finite values.
// The workgroup takes its tile's items ((segment, line) pairs)
// in chunks of CH <= NT: phase 1 gives each of CH threads one item (the walk
// replay, column records into LDS); phase 2 gives each thread one (item,
// column, half) unit of the fills at a time.  The first chunk's loads and
// (256-thread float sum tiles) the tile's current values in `out` are
// requested before the LDS tile is cleared, so their latency overlaps.
// (at least 5 waves per SIMD: the fastest register budget measured)
template <typename T, int K, int OV, int TILE, int SEG, int NT, int CH, bool FAST>
__global__ void __launch_bounds__(NT, 5)
k_tiles(T *__restrict__ out, Geometry g, const int *__restrict__ tile_off, const int2 *__restrict__ pairs,
        const Segment<T> *__restrict__ segs, const LineSetup<T> *__restrict__ setup, T max_val,
        int *__restrict__ flags)
{
    using Acc = typename AccType<T, OV>::type;
    static_assert(OV != 2, "fixed-point sums: k_tiles_fast");
    // LDS pitch TILE: the bank conflicts of the fills (steep lines write one
    // bank from consecutive rows, the two halves of a column share a bank) and
    // of the strided item records cost less than removing them did (a padded
    // pitch and rotated record slots spilled registers at 5 waves per SIMD or
    // dropped to 4)
    constexpr int PITCH = TILE;
    constexpr int LDS_PX = TILE * PITCH;   // LDS words of the tile (pixel (y, x) at y * PITCH + x)
    __shared__ alignas(16) Acc img[LDS_PX];
    uint32_t *const zb = nullptr;   // (zero bits of fixed-point sums: unused here)
    static_assert(CH <= NT, "one phase-1 thread per item");
    __shared__ int32_t rs[CH * SEG + CH];   // + one sink slot per phase-1 lane
    __shared__ T rT[CH * SEG + CH];
    __shared__ T rN[CH * SEG + CH];
    __shared__ FillRec frec[CH];

    const int tile = blockIdx.x;
    // (one round trip for the item range and the error flags: a plan's draw
    // reports errors afterwards and leaves `out` untouched then)
    const int beg = tile_off[tile * LIST_SUBS], end = tile_off[(tile + 1) * LIST_SUBS];
    const int fl = *flags;
    if (fl || beg == end) return;
    const int per_frame = g.ntx * g.nty;
    const int64_t f = tile / per_frame;
    const int r = tile - (int)f * per_frame;
    const int ty = r / g.ntx, tx = r - ty * g.ntx;
    const int X0 = tx * TILE, Y0 = ty * TILE;
    const int X1 = min(X0 + TILE, g.W), Y1 = min(Y0 + TILE, g.H);
    const int tid = threadIdx.x;
    T *fo = out + (f * g.H) * (int64_t)g.W;
    constexpr int V = 4;
    const bool full = (X1 - X0 == TILE) && ((g.W & (V - 1)) == 0) && (((uintptr_t)out & 15) == 0);

    // the tile's current values, for the flush (float sums, 256 threads:
    // 4 float4 per thread), requested first
    constexpr bool PREF = (OV != 1) && sizeof(T) == 4 && NT == 256 && TILE == 64;
    constexpr int PV = PREF ? (TILE * TILE) / (NT * V) : 1;
    float4 pre[PV];
    if constexpr (PREF) {
        if (full) {
#pragma unroll
            for (int j = 0; j < PV; j++) {
                const int i = (tid + j * NT) * V;
                const int y = Y0 + i / TILE, x = X0 + (i % TILE);
                if (y < Y1) {
                    const v4f q = __builtin_nontemporal_load(reinterpret_cast<const v4f *>(fo + (int64_t)y * g.W + x));
                    pre[j] = make_float4(q.x, q.y, q.z, q.w);
                }
            }
        }
    }
    // first chunk's item loads (after the tile's loads, which do not wait on them)
    Segment<T> sg0;
    LineSetup<T> L0;
    if (tid < min(CH, end - beg)) {
        const int2 it = pairs[beg + tid];
        sg0 = segs[it.x];
        L0 = setup[it.y];
    }

    auto clear = [&]() {
        if constexpr (OV != 0 && sizeof(Acc) == 4) {
            // zero words (below every max code / empty fixed-point sum), 16 bytes per store
            static_assert(LDS_PX % 4 == 0, "whole 16-byte stores");
            uint4 *p = reinterpret_cast<uint4 *>(img);
            for (int i = tid; i < LDS_PX / 4; i += NT) p[i] = make_uint4(0u, 0u, 0u, 0u);
        } else {
            for (int i = tid; i < LDS_PX; i += NT) {
                if constexpr (OV == 0) img[i] = Acc(-0.0); // additive identity, keeps -0.0 pixels intact
                else img[i] = Acc(0);                      // below every max code
            }
        }
    };
    clear();

    const T vscale = max_val;
    {
        const int rb = beg, re = end;
        for (int first = rb; first < re; first += CH) {
            const int n = min(CH, re - first);
            // (phase 1 writes only the item records: the first chunk needs no
            // barrier after the clear)
            if (first != beg) __syncthreads();
            // phase 1: replay the walk of one item from its checkpoint and
            // record the centre and errors of every emitted column
            if (tid < n) {
                Segment<T> sg;
                LineSetup<T> L;
                if (first == beg) {
                    sg = sg0;
                    L = L0;
                } else {
                    const int2 it = pairs[first + tid];
                    sg = segs[it.x];
                    L = setup[it.y];
                }
                const int a = L.axis, sa = pick(L.st, a);
                const int c0 = pick(sg.c, a);
                // per-line profiles: the wave's items take their record slots
                // grouped by profile, so the fills of a wave mostly share one
                // (the sums do not depend on the item order but for their rounding)
                int dst = tid;
                if constexpr (K == K_MIXED) {
                    const int kc = (L.kid >= 0 && L.kid < K_TRIANGULAR) ? L.kid : K_TRIANGULAR;
                    const uint64_t below = (1ull << (tid & 63)) - 1ull;
                    int off = 0, rank = 0;
#pragma unroll
                    for (int k = 0; k <= K_TRIANGULAR; k++) {
                        const uint64_t m = __ballot(kc == k);
                        if (kc == k) rank = off + __popcll(m & below);
                        off += __popcll(m);
                    }
                    dst = (tid & ~63) + rank;
                }
                frec[dst] = fill_rec(L, c0, sg.line);
#pragma unroll
                for (int k = 0; k < SEG; k++) rs[dst * SEG + k] = INT_MIN;
                WalkState<T> s;
                s.c[0] = sg.c[0];
                s.c[1] = sg.c[1];
                s.Te = sg.Te;
                s.Ne = sg.Ne;
                // a loop uniform over the wave: lanes whose walk has ended are
                // masked by predicates and store into their sink slot
                bool act = true;
                for (int it = 0; it < 4 * SEG + 16; it++) {
                    act = act && !walk_done(L, s);
                    const int k = (pick(s.c, a) - c0) * sa;
                    act = act && k < sg.ncols;
                    if (__ballot(act) == 0) break;
                    bool nx, ny;
                    walk_next(L, s.Ne, nx, ny);
                    const bool rec = act && ((a == 0) ? nx : ny);
                    const int slot = rec ? dst * SEG + k : CH * SEG + tid;
                    rs[slot] = pick(s.c, 1 - a);
                    rT[slot] = s.Te;
                    rN[slot] = s.Ne;
                    walk_step(L, s, act && nx, act && ny);
                }
                if (act) atomicOr(flags, FLAG_STUCK);   // still walking after the step budget
            }
            __syncthreads();
            // phase 2: one thread per (item, column, half); the centre goes
            // with the half that steps in +st[b] (bresenham.hpp:364-380)
            for (int u = tid; u < n * SEG * 2; u += NT) {
                const int i = u / (2 * SEG), rem = u - i * (2 * SEG);
                const int k = rem >> 1, half = rem & 1;
                const int slot = i * SEG + k;
                const int cs = rs[slot];
                if (cs == INT_MIN) continue;
                const FillRec R = frec[i];
                const int a = R.meta & FR_AXIS, b = 1 - a;
                const int c = R.c0 + ((R.meta & FR_SA) ? k : -k);
                const int s_lo = (a == 0) ? Y0 : X0, s_hi = (a == 0) ? Y1 : X1;
                // LDS stride of the short axis and offset of the long-axis column
                const int sstride = (a == 0) ? PITCH : 1;
                const int cbase = (a == 0) ? (c - X0) : (c - Y0) * PITCH;
                T Te = rT[slot], Ne = rN[slot];
                if constexpr (FAST && sizeof(T) == 4) {
                    if (R.meta & FR_SAFE) {
                        fill_half_fast<K, OV>(img, zb, R, setup[R.line], cs, Te, Ne, half, cbase, sstride, s_lo,
                                              s_hi, (float)vscale);
                        continue;
                    }
                }
                const LineSetup<T> L = setup[R.line];
                auto put = [&](int s, T Te_, T nsq) {
                    T v;
                    if (!pixel_eval<FAST, K>(L, Te_, nsq, vscale, v)) return;
                    tile_put<OV>(img, zb, cbase + (s - s_lo) * sstride, v);
                };
                if (half == 0 && cs >= s_lo && cs < s_hi) put(cs, Te, nsq_of(L, Ne));
                const int sb = pick(L.st, b);
                const int dir = half ? -sb : sb;
                const T tb = pick(L.t, b), nb = pick(L.nv, b);
                const T dT = (dir > 0) ? tb : -tb, dN = (dir > 0) ? nb : -nb;
                int s = cs;
                for (;;) {
                    s += dir;
                    Te += dT;
                    Ne += dN;
                    const T nsq = nsq_of(L, Ne);
                    if (!(nsq < L.w2)) break;
                    if (s >= s_lo && s < s_hi) put(s, Te, nsq);
                    else if ((dir > 0) ? (s >= s_hi) : (s < s_lo)) break;
                }
            }
        }
    }
    __syncthreads();

    // flush: one coalesced read-modify-write of the tile, 4 pixels per access
    // where the tile row lies inside the frame
    if constexpr (PREF) {
        if (full) {
#pragma unroll
            for (int j = 0; j < PV; j++) {
                const int i = (tid + j * NT) * V;
                const int y = Y0 + i / TILE, x = X0 + (i % TILE);
                if (y >= Y1) continue;
                const int li = (i / TILE) * PITCH + (i % TILE);
                float4 ov = pre[j];
                ov.x = (float)((double)ov.x + img[li]);
                ov.y = (float)((double)ov.y + img[li + 1]);
                ov.z = (float)((double)ov.z + img[li + 2]);
                ov.w = (float)((double)ov.w + img[li + 3]);
                *reinterpret_cast<float4 *>(fo + (int64_t)y * g.W + x) = ov;
            }
            return;
        }
    }
    for (int i = tid * V; i < TILE * TILE; i += NT * V) {
        const int y = Y0 + i / TILE, x = X0 + (i % TILE);
        if (y >= Y1) continue;
        T *o = fo + (int64_t)y * g.W + x;
        const int li = (i / TILE) * PITCH + (i % TILE);
        if (full) {
            if constexpr (OV == 0) {
                if constexpr (sizeof(T) == 4) {
                    float4 ov = *reinterpret_cast<float4 *>(o);
                    ov.x = (float)((double)ov.x + img[li]);
                    ov.y = (float)((double)ov.y + img[li + 1]);
                    ov.z = (float)((double)ov.z + img[li + 2]);
                    ov.w = (float)((double)ov.w + img[li + 3]);
                    *reinterpret_cast<float4 *>(o) = ov;
                } else {
                    for (int j = 0; j < V; j++) o[j] = o[j] + img[li + j];
                }
            } else {
                for (int j = 0; j < V; j++) {
                    const Acc e = img[li + j];
                    if (e != Acc(0)) {
                        const T m = ord_dec(e);
                        const T ov = o[j];
                        o[j] = (ov < m) ? m : ov; // std::max(out, value)
                    }
                }
            }
        } else {
            for (int j = 0; j < V; j++) {
                if (x + j >= X1) break;
                if constexpr (OV == 0) {
                    o[j] = (T)((double)o[j] + img[li + j]);
                } else {
                    const Acc e = img[li + j];
                    if (e != Acc(0)) {
                        const T m = ord_dec(e);
                        const T ov = o[j];
                        o[j] = (ov < m) ? m : ov;
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// 5. tile kernel of the float images (fast values; float sums and max)
// ---------------------------------------------------------------------------
// One column half of any line with the full error: the fast path, or for lines
// that are not FR_SAFE the general error estimate of pixel_eval.
template <int K, int OV, typename Acc>
__device__ __forceinline__ void fill_half(Acc *img, uint32_t *zb, const FillRec &R,
                                          const LineSetup<float> *__restrict__ setup, int cs, float Te, float Ne,
                                          int half, int cbase, int sstride, int s_lo, int s_hi, float vscale)
{
    if (R.meta & FR_SAFE) {
        fill_half_fast<K, OV>(img, zb, R, setup[R.line], cs, Te, Ne, half, cbase, sstride, s_lo, s_hi, vscale);
        return;
    }
    const LineSetup<float> G = setup[R.line];
    auto put = [&](int s, float Te_, float nsq) {
        float v;
        if (!pixel_eval<true, K>(G, Te_, nsq, vscale, v)) return;
        tile_put<OV>(img, zb, cbase + (s - s_lo) * sstride, v);
    };
    if (half == 0 && cs >= s_lo && cs < s_hi) put(cs, Te, nsq_of(G, Ne));
    const int sb = (R.meta & FR_SB) ? 1 : -1;
    const int dir = half ? -sb : sb;
    const float dT = (dir > 0) ? R.tb : -R.tb, dN = (dir > 0) ? R.nb : -R.nb;
    int s = cs;
    for (;;) {
        s += dir;
        Te += dT;
        Ne += dN;
        const float nsq = nsq_of(G, Ne);
        if (!(nsq < G.w2)) break;
        if (s >= s_lo && s < s_hi) put(s, Te, nsq);
        else if ((dir > 0) ? (s >= s_hi) : (s < s_lo)) break;
    }
}

// The profile at normal error x = |Ne| sqrt(ea k) (k: interior_scale), for
// pixels with no tangential overshoot: c K(sqrt(u)) with u = Ne^2 ea.
template <int K>
constexpr float interior_scale() { return K == K_GAUSSIAN ? 6.4921276840f : 1.0f; }   // exp(-4.5 u) = 2^(-k u)

template <int K>
__device__ __forceinline__ float interior_value(float x, float c)
{
    if constexpr (K == K_BIWEIGHT) {
        const float m = __builtin_fmaf(-x, x, 1.0f);
        return c * (m * m);
    } else if constexpr (K == K_GAUSSIAN) {
        return c * __builtin_amdgcn_exp2f(-(x * x));
    } else if constexpr (K == K_PARABOLIC) {
        return c * __builtin_fmaf(-x, x, 1.0f);
    } else if constexpr (K == K_RECTANGULAR) {
        return c;
    } else {
        return __builtin_fmaf(-c, __builtin_fabsf(x), c);
    }
}

// What phase 2a of k_tiles_fast needs of an item (see fill_interior).
struct alignas(16) InnerRec {
    float inv;        // 1 / nb: nb is the normal error's change per +1 along the short axis
    float hm, hp;     // half height of the band in steps: decided inside (hm), decided outside (hp)
    float rs;         // sqrt(ea k)
    float dx;         // nb rs
    float cap, far;   // interior columns: cap < Te < far
    int32_t base;     // LDS index of column 0 at short-axis coordinate 0
};

// Fills of one interior column: no pixel of it has a tangential overshoot, and
// |Ne| <= |nb| at its centre.  Away from the centre |N_j| grows with every
// step, so the reference's two half loops emit exactly the pixels j (steps
// along +s) with |N_j| < nlim: those with j in (jc - h, jc + h), jc = -Ne / nb,
// h = nlim / |nb|.  Pixels nearer to an end of that range than a tolerance
// (the error of the estimate and of the reference's own running sums, and the
// 2e-6 that separate the band test from error <= 1) are decided by the
// reference's additions and the exact error (rare); the others need no test, so
// the loop is straight-line code with its count known beforehand.
template <int K, int OV, typename Acc>
__device__ __forceinline__ void fill_interior(Acc *img, uint32_t *zb, const InnerRec &I, const FillRec *rec,
                                              const LineSetup<float> *__restrict__ setup, int cs, float Ne, float jc,
                                              int at, int sstride, int w0, int w1, float vscale)
{
    const float c = fast_scale<K>(0, vscale);
    const float f0 = __builtin_ceilf(jc - I.hm), f1 = __builtin_floorf(jc + I.hm);
    const int j0 = (int)f0, j1 = (int)f1;
    const int a = max(j0, w0);
    const int n = min(j1, w1) - a + 1;
    const float x0 = Ne * I.rs;
    float jf = (float)a;
    Acc *q = img + (at + a * sstride);
    for (Acc *const e = q + max(n, 0) * sstride; q != e; q += sstride) {
        const float v = interior_value<K>(__builtin_fmaf(jf, I.dx, x0), c);
        if constexpr (OV == 2) {
            // (not cut after adding 0.5 inside the value's product, one instruction
            // less: from 2^23 on that sum is rounded itself)
            const uint32_t u = __float2uint_rn(v);
            atomicAdd(q, fast_positive<K>() ? u : max(1u, u));
        } else {
            atomicMax(q, ord_enc(v));
        }
        jf += 1.0f;
    }
    // the undecided pixels next to the band's ends
    const float g0 = __builtin_ceilf(jc - I.hp), g1 = __builtin_floorf(jc + I.hp);
    if (g0 < f0 || g1 > f1) {
        const FillRec R = *rec;
        const LineSetup<float> L = setup[R.line];
        for (int j = (int)g0; j <= (int)g1; j++) {
            if ((j >= j0 && j <= j1) || j < w0 || j > w1) continue;
            float N = Ne;
            const float dN = (j < 0) ? -R.nb : R.nb;
            for (int i = 0; i < abs(j); i++) N += dN;
            if (j != 0 && !(__builtin_fabsf(N) < R.nlim)) continue;
            const float e = err_fast(L, R.LL, R.ea, 0.0f, N);
            if (e <= 1.0f) tile_put<OV>(img, zb, at + j * sstride, fast_value<K>(0, e, c));
        }
    }
}

// One workgroup per tile, NT / 64 independent waves.  A wave takes chunks of up to
// CHW items: phase 1 replays one item's walk per lane (FP32 steps as the
// reference's) and records every column's centre and errors in the wave's own
// LDS area; phase 2a gives each lane one interior column (both halves in one
// loop, no tangent term); phase 2b takes the other columns (within the
// width of a line's end) from a compacted list, one (column, half) per lane,
// with the full error.  Only the tile's accumulator is shared: one barrier
// after the clear and one before the fold, so that one wave's walk replay
// overlaps another's fills.
//
// Bound by vector instruction issue: 64 frames of 2048^2 with 128 000 gaussian
// lines take 0.59 ms (the image alone is 0.46 ms at a copy's rate), 32 of 1024^2
// with 160 000 biweight lines 0.33 ms (175 M wave instructions, 0.28 ms at the
// issue rate), 256 of 1024^2 with 972 000 lines of mixed profiles and 16-column
// segments 2.6 ms (1356 M, 2.2 ms).  With one tested, sequential loop per half column (k_tiles' fills) and
// one wave replaying the walks of the whole workgroup the same took 0.66, 0.60
// and 5.1 ms: 60 % of the instructions were the loop's tests, masks and idle lanes.
//
// FEW: tiles of a few items, whose time is latency.  Half the records and no pixel
// values held beside them, so that five workgroups fit a CU instead of four, and
// only touched pixels are read and written, by the same operations.  20 000 frames of
// 64^2 with a line each: call 138 -> 123 us (max 119 -> 115), 133 (119) with k_tiles'
// fills; of 33 x 33 with two 175 -> 147 (158).
template <int K, int OV, int TILE, int SEG, int NT, int CHW, bool FEW>
__global__ void __launch_bounds__(NT, FEW ? 6 : 4)
k_tiles_fast(float *__restrict__ out, Geometry g, const int *__restrict__ tile_off, const int2 *__restrict__ pairs,
             const Segment<float> *__restrict__ segs, const LineSetup<float> *__restrict__ setup,
             const LineLite *__restrict__ lite, float max_val, int *__restrict__ flags)
{
    static_assert(OV == 1 || OV == 2, "max codes or fixed-point sums");
    static_assert(CHW <= 64, "one lane per item");
    constexpr int NW = NT / 64, PX = TILE * TILE, NREC = CHW * SEG;
    // Rows 4 words apart in the banks: the columns of a steep line add to one x in
    // consecutive rows, which share a bank with a pitch of TILE (160 000 lines of
    // widths 2 to 6: 333 -> 321 us; conflict cycles a third fewer).
    constexpr int PITCH = TILE + 4, LP = TILE * PITCH;
    __shared__ alignas(16) uint32_t img[LP];
    __shared__ uint32_t zb[OV == 2 ? LP / 32 : 1];
    __shared__ WaveCols<NREC> cols[NW];
    __shared__ FillRec frec[NW][CHW];
    __shared__ InnerRec irec[NW][CHW];
    __shared__ uint16_t caps[NW][NREC];

    const int tile = blockIdx.x;
    const int beg = tile_off[tile * LIST_SUBS], end = tile_off[(tile + 1) * LIST_SUBS];
    const int fl = *flags;
    if (fl || beg == end) return;
    int64_t f;
    int tx, ty;
    tile_coords(g, tile, f, tx, ty);
    const int X0 = tx * TILE, Y0 = ty * TILE;
    const int X1 = min(X0 + TILE, g.W), Y1 = min(Y0 + TILE, g.H);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *const to = out + ((f * g.H + Y0) * (int64_t)g.W + X0);   // the tile's first pixel
    const bool full = (X1 - X0 == TILE) && ((g.W & 3) == 0) && (((uintptr_t)out & 15) == 0);

    // the tile's current values, requested first (sums): four consecutive
    // pixels per load where rows allow it, else one (clamped into the frame:
    // pixels outside it are not stored)
    constexpr int PP = PX / NT;   // pixels per thread
    constexpr bool PREF = OV == 2 && PP <= 16 && PP % 4 == 0 && !FEW;
    float pre[PREF ? PP : 1];
    if constexpr (PREF) {
        if (full) {
#pragma unroll
            for (int j = 0; j < PP / 4; j++) {
                const int i = (tid + j * NT) * 4;
                const int y = min(i / TILE, Y1 - Y0 - 1);
                const v4f q = __builtin_nontemporal_load(
                    reinterpret_cast<const v4f *>(to + ((int64_t)y * g.W + (i % TILE))));
                pre[4 * j] = q.x;
                pre[4 * j + 1] = q.y;
                pre[4 * j + 2] = q.z;
                pre[4 * j + 3] = q.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < PP; j++) {
                const int i = tid + j * NT;
                const int y = min(i / TILE, Y1 - Y0 - 1), x = min(i % TILE, X1 - X0 - 1);
                pre[j] = __builtin_nontemporal_load(to + ((int64_t)y * g.W + x));
            }
        }
    }

    // chunks of a round of n items: a multiple of the wave count, of equal
    // size, so that every wave makes the same number of turns
    int turns, size;
    auto split = [&](int n) {
        turns = (n + NW * CHW - 1) / (NW * CHW);
        size = (n + turns * NW - 1) / (turns * NW);
    };
    split((OV == 2) ? min(FIX_ROUND, end - beg) : end - beg);
    Segment<float> sg;
    LineLite L;
    auto take = [&](const int2 &it) {
        sg = segs[it.x];
        L = lite[it.y];
    };
    // (lanes without an item load the list's last)
    take(pairs[min(beg + wave * size + lane, end - 1)]);
    auto clear = [&]() {
        uint4 *p = reinterpret_cast<uint4 *>(img);
        for (int i = tid; i < LP / 4; i += NT) p[i] = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (OV == 2)
            for (int i = tid; i < LP / 32; i += NT) zb[i] = 0u;
    };
    clear();

    WaveCols<NREC> &wK = cols[wave];
    FillRec *const wR = frec[wave];
    InnerRec *const wI = irec[wave];
    uint16_t *const wC = caps[wave];
    const uint64_t below = (1ull << lane) - 1ull;

    for (int rb = beg, re; rb < end; rb = re) {
        re = (OV == 2) ? rb + min(FIX_ROUND, end - rb) : end;
        const int F = (OV == 2) ? __clz(re - rb) : 0;
        const float vscale = (OV == 2) ? __int_as_float((127 + F) << 23) : max_val;
        if (rb != beg) {
            split(re - rb);
            take(pairs[min(rb + wave * size + lane, end - 1)]);
            clear();
        }
        for (int t = 0; t < turns; t++) {
            const int first = rb + (t * NW + wave) * size;
            const int n = max(0, min(size, re - first));
            const int2 np = pairs[min(first + NW * size + lane, end - 1)];   // the next turn's items
            // phase 1
            {
                const int meta = L.meta;
                const bool ax = meta & FR_AXIS;
                const float t0 = L.t[0], t1 = L.t[1];
                int dst = lane;
                if constexpr (K == K_MIXED) {
                    // record slots grouped by profile, so that the fills of a
                    // wave mostly share one
                    const int kid = lane < n ? ((meta >> 8) & 0xff) : K_MIXED;
                    int off = 0;
#pragma unroll
                    for (int k = 0; k <= K_MIXED; k++) {
                        const uint64_t m = __ballot(kid == k);
                        if (kid == k) dst = off + __popcll(m & below);
                        off += __popcll(m);
                    }
                }
                if (lane < n) {
                    const float nb = ax ? t1 : -t0, na = __builtin_fabsf(nb);
                    FillRec R;
                    R.LL = L.LL;
                    R.ea = L.ea;
                    R.nlim = L.nlim;
                    R.tb = ax ? t0 : t1;
                    R.nb = nb;
                    R.c0 = ax ? sg.c[0] : sg.c[1];
                    R.line = sg.line;
                    R.meta = meta | (sg.ncols << 16);
                    wR[dst] = R;
                    InnerRec I;
                    I.inv = __builtin_amdgcn_rcpf(nb);
                    const float h = L.nlim * __builtin_fabsf(I.inv), tol = h * (8e-6f + 3e-7f * h);
                    I.hm = h - tol;
                    I.hp = h + tol;
                    const int kid = (K == K_MIXED) ? ((meta >> 8) & 0xff) : K;
                    I.rs = __builtin_amdgcn_sqrtf(
                        L.ea * (kid == K_GAUSSIAN ? interior_scale<K_GAUSSIAN>() : interior_scale<K_BIWEIGHT>()));
                    I.dx = nb * I.rs;
                    // (thicker lines: the running sums drift further from the estimate)
                    I.cap = ((meta & FR_SAFE) && L.nlim < 64.0f * na) ? L.cap : __builtin_inff();
                    I.far = L.LL - L.cap;
                    I.base = ax ? (sg.c[1] - Y0) * PITCH - X0 : (sg.c[0] - X0) - Y0 * PITCH;
                    wI[dst] = I;
                    if (!replay_columns<SEG>(wK, L, sg, dst * SEG, sg.ncols)) atomicOr(flags, FLAG_STUCK);
                }
            }
            take(np);
            wave_sync();
            if (t == 0) __syncthreads();   // the cleared tile
            // phase 2a
            int ncap = 0;
            for (int u0 = 0; u0 < n * SEG; u0 += 64) {
                const int u = u0 + lane, i = u / SEG, k = u % SEG;
                bool cap = false;
                if (u < n * SEG) {
                    const int meta = wR[i].meta;
                    if (k < (meta >> 16)) {
                        const InnerRec I = wI[i];
                        const float Te = wK.T[u], Ne = wK.N[u];
                        const float jc = -Ne * I.inv;
                        cap = !(Te > I.cap && Te < I.far && __builtin_fabsf(jc) <= 1.0f);
                        if (!cap) {
                            const int cs = wR[i].c0 + wK.centre(u);
                            const bool ax = meta & FR_AXIS;
                            const int kk = (meta & FR_SA) ? k : -k;
                            const int sst = ax ? 1 : PITCH;
                            const int at = I.base + kk * (ax ? PITCH : 1) + cs * sst;
                            const int w0 = (ax ? X0 : Y0) - cs, w1 = (ax ? X1 : Y1) - 1 - cs;
                            if constexpr (K == K_MIXED) {
#define CBX_INNER(KK) fill_interior<KK, OV>(img, zb, I, wR + i, setup, cs, Ne, jc, at, sst, w0, w1, vscale)
                                switch ((meta >> 8) & 0xff) {
                                case K_BIWEIGHT: CBX_INNER(K_BIWEIGHT); break;
                                case K_GAUSSIAN: CBX_INNER(K_GAUSSIAN); break;
                                case K_PARABOLIC: CBX_INNER(K_PARABOLIC); break;
                                case K_RECTANGULAR: CBX_INNER(K_RECTANGULAR); break;
                                default: CBX_INNER(K_TRIANGULAR);
                                }
#undef CBX_INNER
                            } else {
                                fill_interior<K, OV>(img, zb, I, wR + i, setup, cs, Ne, jc, at, sst, w0, w1, vscale);
                            }
                        }
                    }
                }
                const uint64_t cm = __ballot(cap);
                if (cap) wC[ncap + __popcll(cm & below)] = (uint16_t)u;
                ncap += __popcll(cm);
            }
            wave_sync();
            // phase 2b
            for (int u = lane; u < 2 * ncap; u += 64) {
                const int slot = wC[u >> 1], half = u & 1;
                const int i = slot / SEG, k = slot % SEG;
                const FillRec R = wR[i];
                const int cs = R.c0 + wK.centre(slot);
                const int a = R.meta & FR_AXIS;
                const int kk = (R.meta & FR_SA) ? k : -k;
                const int s_lo = a ? X0 : Y0, s_hi = a ? X1 : Y1;
                const int sstride = a ? 1 : PITCH;
                const int cbase = wI[i].base + kk * (a ? PITCH : 1) + s_lo * sstride;
                fill_half<K, OV>(img, zb, R, setup, cs, wK.T[slot], wK.N[slot], half, cbase, sstride, s_lo, s_hi, vscale);
            }
            wave_sync();
        }
        __syncthreads();
        if constexpr (OV == 2) {
            // fold the round into the pixel values (registers or `out`)
            const double scale = ldexp((double)max_val, -F);
            const float zero = max_val * 0.0f, p2 = __int_as_float((127 - F) << 23);   // 2^-F, F <= 31
            if constexpr (FEW) {
                // the touched pixels only, a batch's loads before its stores
                constexpr int B = PP < 8 ? PP : 8;
                int t0 = tid;
                asm("" : "+v"(t0));   // (addresses are made here, not kept in registers through the round)
#pragma unroll 1
                for (int i0 = t0; i0 < (Y1 - Y0) * TILE; i0 += B * NT) {
                    float o[B];
                    uint32_t acc[B], z[B];
#pragma unroll
                    for (int j = 0; j < B; j++) {
                        const int i = i0 + j * NT, y = i / TILE, x = i % TILE, li = y * PITCH + x;
                        acc[j] = img[li];
                        z[j] = (zb[li >> 5] >> (li & 31)) & 1u;
                        // (pixels outside the frame are never touched)
                        o[j] = (acc[j] | z[j]) ? to[(int64_t)y * g.W + x] : 0.0f;
                    }
#pragma unroll
                    for (int j = 0; j < B; j++) {
                        const int i = i0 + j * NT, y = i / TILE, x = i % TILE;
                        if (!(acc[j] | z[j])) continue;
                        const double add = acc[j] ? (double)acc[j] * scale : (double)zero;
                        to[(int64_t)y * g.W + x] =
                            full ? fold_fix(o[j], acc[j], z[j], p2, max_val, zero) : (float)((double)o[j] + add);
                    }
                }
            } else if (PREF && full) {
                // all LDS reads first (4 pixels and their zero bits per read),
                // then branch-free updates
                const uint32_t l4 = (uint32_t)tid * 4 / TILE * PITCH + (uint32_t)tid * 4 % TILE;
                uint4 acc[PP / 4];
                uint32_t zw[PP / 4];
#pragma unroll
                for (int j = 0; j < PP / 4; j++) {
                    constexpr int ROWS = NT * 4 / TILE * PITCH;
                    static_assert(!PREF || ROWS % 32 == 0, "whole words of zero bits");
                    acc[j] = *reinterpret_cast<const uint4 *>(&img[l4 + j * ROWS]);
                    zw[j] = zb[l4 / 32 + j * (ROWS / 32)] >> (l4 % 32);
                }
#pragma unroll
                for (int j = 0; j < PP / 4; j++) {
                    pre[4 * j] = fold_fix(pre[4 * j], acc[j].x, zw[j] & 1u, p2, max_val, zero);
                    pre[4 * j + 1] = fold_fix(pre[4 * j + 1], acc[j].y, zw[j] & 2u, p2, max_val, zero);
                    pre[4 * j + 2] = fold_fix(pre[4 * j + 2], acc[j].z, zw[j] & 4u, p2, max_val, zero);
                    pre[4 * j + 3] = fold_fix(pre[4 * j + 3], acc[j].w, zw[j] & 8u, p2, max_val, zero);
                }
            } else if (PREF) {
                uint32_t acc[PP], z[PP];
#pragma unroll
                for (int j = 0; j < PP; j++) {
                    const uint32_t li = (uint32_t)tid / TILE * PITCH + (uint32_t)tid % TILE + j * (NT / TILE * PITCH);
                    acc[j] = img[li];
                    z[j] = (zb[li >> 5] >> (li & 31)) & 1u;
                }
#pragma unroll
                for (int j = 0; j < PP; j++) {
                    const double add = acc[j] ? (double)acc[j] * scale : (double)zero;
                    const float v = (float)((double)pre[j] + add);
                    pre[j] = (acc[j] | z[j]) ? v : pre[j];
                }
            } else {
                bool has;
                for (int i = tid; i < PX; i += NT) {
                    const int y = i / TILE, x = i % TILE;
                    if (y >= Y1 - Y0 || x >= X1 - X0) continue;
                    const double add = fix_value(img[y * PITCH + x], zb, y * PITCH + x, scale, max_val, has);
                    float *o = to + ((int64_t)y * g.W + x);
                    if (has) *o = (float)((double)*o + add);
                }
            }
            if (re < end) __syncthreads();   // before the next round clears the tile
        }
    }
    if constexpr (PREF) {
        // written once per draw: non-temporal
        if (full) {
#pragma unroll
            for (int j = 0; j < PP / 4; j++) {
                const int i = (tid + j * NT) * 4;
                const v4f q = {pre[4 * j], pre[4 * j + 1], pre[4 * j + 2], pre[4 * j + 3]};
                if (i / TILE < Y1 - Y0)
                    __builtin_nontemporal_store(q, reinterpret_cast<v4f *>(to + ((int64_t)(i / TILE) * g.W + (i % TILE))));
            }
        } else {
#pragma unroll
            for (int j = 0; j < PP; j++) {
                const int i = tid + j * NT;
                if (i / TILE < Y1 - Y0 && i % TILE < X1 - X0)
                    __builtin_nontemporal_store(pre[j], to + ((int64_t)(i / TILE) * g.W + (i % TILE)));
            }
        }
    } else if constexpr (OV == 1) {
        // every value is requested before any is used; std::max(out, value)
        constexpr int B = FEW ? (PP < 8 ? PP : 8) : (PP < 16 ? PP : 16);
        for (int i0 = tid; i0 < (FEW ? (Y1 - Y0) * TILE : PX); i0 += B * NT) {
            float o[B];
            uint32_t e[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int i = i0 + j * NT;
                const int y = i / TILE, x = i % TILE;
                e[j] = img[y * PITCH + x];
                if constexpr (FEW) o[j] = e[j] ? to[(int64_t)y * g.W + x] : 0.0f;
                else o[j] = to[(int64_t)min(y, Y1 - Y0 - 1) * g.W + min(x, X1 - X0 - 1)];
            }
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int i = i0 + j * NT;
                const float m = ord_dec(e[j]);
                // (pixels outside the frame are never drawn: e = 0)
                if (e[j] && o[j] < m) to[(int64_t)(i / TILE) * g.W + (i % TILE)] = m;
            }
        }
    }
}

template <int K, int OV, int TILE, int SEG>
static void launch_fast(float *out, const SegmentPlan<float> &P, float max_val, int threads, int chunk, bool,
                        hipStream_t st)
{
#define CBX_TILES_FAST(NT, CHW, FEW)                                                                            \
    k_tiles_fast<K, OV, TILE, SEG, NT, CHW, FEW><<<(unsigned)P.n_tiles, NT, 0, st>>>(                               \
        out, P.g, P.tile_off.ptr, P.pairs.ptr, P.segs.ptr, P.setup.ptr, P.lite.ptr, max_val, P.flags.ptr)
    // 256 records per wave: four workgroups' areas fit a CU's LDS and the tile's few items spread over
    // its waves (64 frames of 2048^2, seg 8: 24 / 32 / 48 items 0.604 / 0.592 / 0.721 ms; 256 of 1024^2,
    // seg 16: 8 / 16 / 24 / 32 items 3.72 / 2.80 / 3.07 / 2.89 ms)
    if (threads == 64) CBX_TILES_FAST(64, 64, false);
    else if (threads == 128) CBX_TILES_FAST(128, 32, false);
    else if (chunk == 64 && few_items(P)) CBX_TILES_FAST(256, 128 / SEG, true);
    else if (chunk == 64) CBX_TILES_FAST(256, (SEG == 8 ? 32 : 16), false);
    else CBX_TILES_FAST(256, (SEG == 8 ? 64 : 32), false);
#undef CBX_TILES_FAST
}

template <typename T, int K, int OV, int TILE, int SEG>
static void launch_tiles(T *out, const SegmentPlan<T> &P, T max_val, int threads, int chunk, bool fast,
                         hipStream_t st)
{
#define CBX_TILES(NT, CH, FST)                                                                                  \
    k_tiles<T, K, OV, TILE, SEG, NT, CH, FST><<<(unsigned)P.n_tiles, NT, 0, st>>>(                             \
        out, P.g, P.tile_off.ptr, P.pairs.ptr, P.segs.ptr, P.setup.ptr, max_val, P.flags.ptr)
    if constexpr (sizeof(T) == 4) {   // (the values of doubles are always exact)
        if (fast) {
            if (threads == 64) CBX_TILES(64, 64, true);
            else if (threads == 128) CBX_TILES(128, 64, true);
            else if (chunk == 64) CBX_TILES(256, 64, true);
            else CBX_TILES(256, 256, true);
            return;
        }
    }
    if (threads == 64) CBX_TILES(64, 64, false);
    else if (threads == 128) CBX_TILES(128, 64, false);
    else if (chunk == 64) CBX_TILES(256, 64, false);
    else CBX_TILES(256, 256, false);
#undef CBX_TILES
}

template <typename T, int K>
void run_tiles_profile(T *out, const SegmentPlan<T> &P, T max_val, int overlap, const cbx_draw_opts *opts,
                       hipStream_t st)
{
    const int threads = (opts && opts->threads) ? opts->threads : 256;
    const bool fast = !(opts && opts->exact_values);
    const int chunk = (opts && opts->chunk) ? opts->chunk : 64;
    const Geometry &g = P.g;
#define CBX_SHAPE(FN, ...)                                                                                      \
    ((g.tile == 64) ? ((g.seg == 16) ? FN<__VA_ARGS__, 64, 16> : FN<__VA_ARGS__, 64, 8>)                        \
                    : ((g.seg == 16) ? FN<__VA_ARGS__, 32, 16> : FN<__VA_ARGS__, 32, 8>))(                      \
        out, P, max_val, threads, chunk, fast, st)
    // k_tiles_fast takes max_val out of the sum and out of the profile's
    // differences: not where it is no finite number (inf * 0 and inf - inf are
    // NaN, where max_val * K(x) is inf)
    if constexpr (sizeof(T) == 4) {
        if (fast && std::isfinite(max_val)) {
            if (overlap == 0) CBX_SHAPE(launch_fast, K, 2);
            else CBX_SHAPE(launch_fast, K, 1);
            return;
        }
    }
    if (overlap == 0) CBX_SHAPE(launch_tiles, T, K, 0);
    else CBX_SHAPE(launch_tiles, T, K, 1);
#undef CBX_SHAPE
}

template void run_tiles_profile<float, CBX_PROFILE>(float *, const SegmentPlan<float> &, float, int,
                                                    const cbx_draw_opts *, hipStream_t);
template void run_tiles_profile<double, CBX_PROFILE>(double *, const SegmentPlan<double> &, double, int,
                                                     const cbx_draw_opts *, hipStream_t);

} // namespace cbx
