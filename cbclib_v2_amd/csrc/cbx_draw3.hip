// 3D lines on gfx950: draw_lines and accumulate_lines for rows of 7
// (x0, y0, z0, x1, y1, z1, width) into volumes (..., D, H, W).
//
// The pixel walk is the reference's draw_line_3d (cbclib_v2/_src/src/
// bresenham.hpp:389-430) on BresenhamPlotter<T, 3> / LineIterator<T, 3>
// (118-348): a tangent error and one normal error per axis pair (0,1),
// (0,2), (1,2), the three-axis Bresenham step with the minimal-|error|
// choice per pair, and at every long-axis step the orthogonal plane filled
// in four quadrants by a 2D walk with single-axis rays.  Every value is
// accumulated with the reference's FP32 (or FP64) additions in its order, and
// divisions and square roots are IEEE (-fhip-fp32-correctly-rounded-divide-
// sqrt), so the emitted pixel set and the per-pixel values are the
// reference's exactly.
//
// A draw records every line's planes (k_walk3_main, a lane per line) and fills
// them (k_fill3, four lanes per plane); above MAX_PLANES planes, and for
// accumulate_lines with different overlaps, four lanes walk a line instead
// (each replays the main-axis walk and fills one quadrant of every orthogonal
// plane; the first also emits the main-axis pixels).  Pixels are applied to
// `out` with global atomics (add for sum, integer max of the bits for max): sums land
// in no fixed order (within float rounding of the single-threaded reference),
// max is exact.  A validation pass runs first, so a call that fails leaves
// `out` untouched.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <string>
#include <type_traits>

#include "cbx_core.hpp"
#include "cbx_host.hpp"

namespace cbx {

constexpr int D3_NT = 128;
constexpr double MAX_VISITS3 = double(int64_t(1) << 30);
constexpr int64_t MAX_PLANES = int64_t(1) << 23;   // recorded planes of a two-phase draw (256 / 384 MiB)

template <typename T>
struct Iter3 {
    int64_t step[3], cur[3];
    bool next[3];
    T te, ne[3];
};

// pair q of UniquePairs<3>: (0,1), (0,2), (1,2)
__device__ __forceinline__ int pair_a(int q) { return q == 2 ? 1 : 0; }
__device__ __forceinline__ int pair_b(int q) { return q == 0 ? 1 : 2; }

// The constants of one line (BresenhamPlotter<T, 3>(line, ceil(w) + 1)).
template <typename T>
struct Line3 {
    T p0[3], t[3], nrm[3][3];
    T len, w2;
    int axis;
    int64_t step[3], m0[3], m1[3];
    int64_t ray_cap;   // steps of one plane ray: at most 2 sqrt(3) (w + 2) for a ray that leaves the ellipse
};

// 0: draws nothing; 1: ready; -1: the walk is longer than MAX_WALK or leaves
// the coordinate range (FLAG_LONG)
template <typename T>
__device__ int line3_setup(const T *ln, Line3<T> &L)
{
    T p1[3];
    for (int i = 0; i < 3; i++) {
        L.p0[i] = ln[i];
        p1[i] = ln[3 + i];
        L.t[i] = p1[i] - L.p0[i];
    }
    const T w = ln[6];
    for (int q = 0; q < 3; q++) {
        const int a = pair_a(q), b = pair_b(q);
        for (int i = 0; i < 3; i++) L.nrm[q][i] = T(0);
        L.nrm[q][a] = p1[b] - L.p0[b];
        L.nrm[q][b] = L.p0[a] - p1[a];
    }
    // error() is +inf for w <= 0, and a NaN never compares true
    if (!(w > T(0))) return 0;
    T mag = T(0);
    for (int i = 0; i < 3; i++) mag += L.t[i] * L.t[i];
    L.len = m_sqrt(mag);
    if (!(L.len > T(0)) || !__builtin_isfinite(L.len) || !__builtin_isfinite(w)) return 0;
    for (int i = 0; i < 3; i++)
        if (!__builtin_isfinite(L.p0[i]) || !__builtin_isfinite(p1[i])) return 0;
    // the first largest |t| (selects, not indexing: the arrays stay in registers)
    int axis = 0;
    T tmax = m_abs(L.t[0]);
    if (tmax < m_abs(L.t[1])) {
        axis = 1;
        tmax = m_abs(L.t[1]);
    }
    if (tmax < m_abs(L.t[2])) axis = 2;
    L.axis = axis;
    const long offset = (long)(m_ceil(w) + T(1));
    T tau[3];
    for (int i = 0; i < 3; i++) tau[i] = L.t[i] / L.len;
    const T tau_ax = (axis == 0) ? tau[0] : ((axis == 1) ? tau[1] : tau[2]);
    const T sc = m_abs((T)offset / tau_ax);
    for (int i = 0; i < 3; i++) {
        L.step[i] = (p1[i] >= L.p0[i]) ? 1 : -1;
        const T a0 = m_round(L.p0[i] - sc * tau[i]), a1 = m_round(p1[i] + sc * tau[i]);
        if (!(m_abs(a0) < T(MAX_COORD)) || !(m_abs(a1) < T(MAX_COORD))) return -1;
        L.m0[i] = (int64_t)a0;
        L.m1[i] = (int64_t)a1 + L.step[i];
    }
    const int64_t span = (axis == 0) ? L.m1[0] - L.m0[0] : ((axis == 1) ? L.m1[1] - L.m0[1] : L.m1[2] - L.m0[2]);
    if (span > MAX_WALK || span < -MAX_WALK) return -1;
    // one lane walks the whole line: at most MAX_VISITS3 pixel visits
    // (about 5.4 w^2 per plane: the ellipse of half-axes w and <= sqrt(3) w)
    const double wc = (double)m_ceil(w) + 2.0;
    if ((double)(span < 0 ? -span : span) * 8.0 * wc * wc > MAX_VISITS3) return -1;
    L.w2 = w * w;
    L.ray_cap = 8 * (int64_t)wc + 64;
    return 1;
}

// LineIterator::update: the next steps from the minimal-|error| choice of
// every pair of moving axes (NormalError::is_next)
template <typename T>
__device__ __forceinline__ void it3_update(const Line3<T> &L, Iter3<T> &it)
{
    for (int i = 0; i < 3; i++) it.next[i] = it.step[i] != 0;
    for (int q = 0; q < 3; q++) {
        const int a = pair_a(q), b = pair_b(q);
        if (!(it.step[a] && it.step[b])) continue;
        const T ex = it.ne[q] + (T)it.step[a] * L.nrm[q][a];
        const T ey = it.ne[q] + (T)it.step[b] * L.nrm[q][b];
        const T exy = ex + (T)it.step[b] * L.nrm[q][b];
        bool f, s;
        if (m_abs(ey) < m_abs(ex)) {
            f = m_abs(exy) < m_abs(ey);
            s = true;
        } else {
            f = true;
            s = m_abs(exy) < m_abs(ex);
        }
        it.next[a] = it.next[a] && f;
        it.next[b] = it.next[b] && s;
    }
}

// LineIterator::increment: the tangent error and the errors of the pairs
// containing the axis
template <typename T>
__device__ __forceinline__ void it3_inc(const Line3<T> &L, Iter3<T> &it, int64_t x, int ax)
{
    it.cur[ax] += x;
    it.te += (T)x * L.t[ax];
    for (int q = 0; q < 3; q++)
        if (pair_a(q) == ax || pair_b(q) == ax) it.ne[q] += (T)x * L.nrm[q][ax];
}

template <typename T>
__device__ __forceinline__ void it3_advance(const Line3<T> &L, Iter3<T> &it)
{
    for (int i = 0; i < 3; i++)
        if (it.next[i]) it3_inc(L, it, it.step[i], i);
    it3_update(L, it);
}

// BresenhamPlotter::normal_error: sum of the squared normal errors, each
// std::pow(T, 2) in double, accumulated into T
template <typename T>
__device__ __forceinline__ T it3_nerr(const Line3<T> &L, const Iter3<T> &it)
{
    T e = T(0);
    for (int q = 0; q < 3; q++) {
        const double v = (double)(it.ne[q] / L.len);
        e = (T)((double)e + v * v);
    }
    return e;
}

// BresenhamPlotter::error: (tangent term^2 + normal error) / w^2
template <typename T>
__device__ __forceinline__ T it3_err(const Line3<T> &L, const Iter3<T> &it)
{
    const T a = -it.te, b = it.te - L.len * L.len;
    const T m = (a < b) ? b : a;
    const T at = (m < T(0)) ? T(0) : m;
    const double qt = (double)(at / L.len);
    return (T)((qt * qt + (double)it3_nerr(L, it)) / (double)L.w2);
}

// draw_line_3d: emit(xyz, error) for every pixel the reference hands to its
// callback, in its order.  Every loop has a step cap that a walk in exact
// arithmetic never reaches (the main walk moves one of its axes towards m1 at
// every step; a plane ray moves monotonically through the ellipse of points
// within w of the line); a walk whose float errors stop changing hits it,
// sets FLAG_STUCK and stops.
//
// The long axis is a template argument, so that every array index below is a
// compile-time constant once the loops are unrolled and the iterator state
// stays in registers.

// the main iterator at m0 (LineIterator's constructor)
template <typename T>
__device__ __forceinline__ void it3_start(const Line3<T> &L, Iter3<T> &it)
{
    T d[3];
    for (int i = 0; i < 3; i++) {
        it.step[i] = L.step[i];
        it.cur[i] = L.m0[i];
        d[i] = (T)L.m0[i] - L.p0[i];
    }
    it.te = T(0);
    for (int i = 0; i < 3; i++) it.te += L.t[i] * d[i];
    for (int q = 0; q < 3; q++) {
        it.ne[q] = T(0);
        for (int i = 0; i < 3; i++) it.ne[q] += L.nrm[q][i] * d[i];
    }
    it3_update(L, it);
}

// The main loop: plane(it) for every iterator state whose long-axis step is
// taken (the planes draw_line_3d fills).  False if the step cap was hit.
template <int AXIS, typename T, typename Plane>
__device__ __forceinline__ bool walk3_main(const Line3<T> &L, int *flags, Plane &plane)
{
    Iter3<T> it;
    it3_start(L, it);
    int64_t main_cap = 64;
    for (int i = 0; i < 3; i++) main_cap += (L.m1[i] - L.m0[i]) * L.step[i];
    for (int64_t n = 0; !(it.cur[0] == L.m1[0] || it.cur[1] == L.m1[1] || it.cur[2] == L.m1[2]); n++) {
        if (n == main_cap) {
            atomicOr(flags, FLAG_STUCK);
            return false;
        }
        if (it.next[AXIS]) plane(it);
        it3_advance(L, it);
    }
    return true;
}

// Quadrant i of the plane through the main iterator state `it`: a 2D walk
// away from the line with single-axis rays from each of its pixels.
template <int AXIS, typename T, typename Emit>
__device__ __forceinline__ bool fill3_quadrant(const Line3<T> &L, const Iter3<T> &it, int i, int *flags, Emit &emit)
{
    constexpr int axis = AXIS, ax1 = (AXIS + 1) % 3, ax2 = (AXIS + 2) % 3;
    Iter3<T> xy = it;
    xy.step[axis] = 0;                                    // collapse(iter, axis)
    it3_update(L, xy);
    if (i & 1) xy.step[ax1] = -xy.step[ax1];              // flip
    if (i >> 1) xy.step[ax2] = -xy.step[ax2];
    it3_update(L, xy);
    const int mv = ((i & 1) ^ (i >> 1)) ? ax2 : ax1;     // move(axis(1 + ...))
    if (mv == ax1) it3_inc(L, xy, xy.step[ax1], ax1);
    else it3_inc(L, xy, xy.step[ax2], ax2);
    it3_update(L, xy);
    for (int64_t r = 0; it3_nerr(L, xy) < L.w2; it3_advance(L, xy), r++) {
        if (r == L.ray_cap) {
            atomicOr(flags, FLAG_STUCK);
            return false;
        }
        emit(xy.cur, it3_err(L, xy));
#pragma unroll
        for (int j = 1; j < 3; j++) {
            const int aj = (axis + j) % 3;
            if (!xy.next[aj]) continue;
            Iter3<T> x = xy;
            x.step[aj] = 0;                               // collapse(iter_xy, axis(j))
            it3_update(L, x);
            it3_advance(L, x);
            for (int64_t q = 0; it3_nerr(L, x) < L.w2; it3_advance(L, x), q++) {
                if (q == L.ray_cap) {
                    atomicOr(flags, FLAG_STUCK);
                    return false;
                }
                emit(x.cur, it3_err(L, x));
            }
        }
    }
    return true;
}

// the whole walk (quad = -1) or the main-axis pixels (quad 0 only) and the
// fills of one quadrant of every plane (quad = 0..3)
template <int AXIS, typename T, typename Emit>
__device__ __forceinline__ void walk3_axis(const Line3<T> &L, int quad, int *flags, Emit &emit)
{
    bool ok = true;
    auto plane = [&](const Iter3<T> &it) {
        if (!ok) return;
        if (quad <= 0) emit(it.cur, it3_err(L, it));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (quad >= 0 && i != quad) continue;
            if (ok) ok = fill3_quadrant<AXIS>(L, it, i, flags, emit);
        }
    };
    walk3_main<AXIS>(L, flags, plane);
}

template <typename T, typename Emit>
__device__ void walk3(const Line3<T> &L, int quad, int *flags, Emit &&emit)
{
    if (L.axis == 0) walk3_axis<0>(L, quad, flags, emit);
    else if (L.axis == 1) walk3_axis<1>(L, quad, flags, emit);
    else walk3_axis<2>(L, quad, flags, emit);
}

// A recorded plane: the main iterator's errors and position (its steps are
// the line's, its next flags follow from them).  line < 0: unused slot.
template <typename T>
struct PlaneState {
    T te, ne[3];
    int32_t cur[3];
    int32_t line;
};

template <typename T>
__device__ __forceinline__ void it3_from(const Line3<T> &L, const PlaneState<T> &ps, Iter3<T> &it)
{
    for (int i = 0; i < 3; i++) {
        it.step[i] = L.step[i];
        it.cur[i] = ps.cur[i];
        it.ne[i] = ps.ne[i];
    }
    it.te = ps.te;
    it3_update(L, it);
}

// *p = std::max(*p, v) (replaced only if *p < v), or *p += v.  Once *p < v, *p can
// only be replaced by other voxels' values, so the maximum may be one of integers
// that nobody waits for: of the bits as signed numbers for v >= 0 (every negative
// value is a smaller one), the minimum of the unsigned bits for v < 0 (every
// value above it is a smaller one).  50 000 lines of widths 1 to 3, max: 603 us with a
// compare-and-swap loop after the value is known, 465 so.
__device__ __forceinline__ float value_now(const float *p)
{
    return __uint_as_float(__hip_atomic_load((const unsigned int *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

__device__ __forceinline__ double value_now(const double *p)
{
    return __longlong_as_double(
        (long long)__hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// (now: value_now(p), loaded early, for OV = 1)
template <int OV>
__device__ __forceinline__ void apply_atomic(float *p, float v, float now)
{
    if (OV == 0) {
        atomicAdd(p, v);
    } else if (now < v) {
        const int b = __float_as_int(v);
        if (b >= 0) atomicMax((int *)p, b);
        else atomicMin((unsigned int *)p, (unsigned int)b);
    }
}

template <int OV>
__device__ __forceinline__ void apply_atomic(double *p, double v, double now)
{
    if (OV == 0) {
        atomicAdd(p, v);
    } else if (now < v) {
        const long long b = __double_as_longlong(v);
        if (b >= 0) atomicMax((long long *)p, b);
        else atomicMin((unsigned long long *)p, (unsigned long long)b);
    }
}

template <int OV, typename T>
__device__ __forceinline__ void apply_atomic(T *p, T v)
{
    apply_atomic<OV>(p, v, (OV == 1) ? value_now(p) : v);
}

struct Vol3 {
    int64_t n_frames, D, H, W;
};

// validation: frame of every line in range, walks of bounded length
template <typename T, typename I>
__global__ void __launch_bounds__(D3_NT)
k_check3(const T *__restrict__ lines, int64_t n_lines, const I *__restrict__ idxs, Vol3 v, int *__restrict__ flags)
{
    const int64_t i = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (i >= n_lines) return;
    if (idxs && (idxs[i] < 0 || (int64_t)idxs[i] >= v.n_frames)) atomicOr(flags, FLAG_INDEX);
    Line3<T> L;
    if (line3_setup(lines + 7 * i, L) < 0) atomicOr(flags, FLAG_LONG);
}

template <typename T, typename I, int K, int OV>
__global__ void __launch_bounds__(D3_NT)
k_draw3(T *__restrict__ out, const T *__restrict__ lines, int64_t n_lines, const I *__restrict__ idxs, Vol3 v, T max_val,
        int *__restrict__ flags)
{
    const int64_t u = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (u >= 4 * n_lines) return;
    const int64_t i = u >> 2;
    Line3<T> L;
    if (line3_setup(lines + 7 * i, L) != 1) return;
    const int64_t f = idxs ? (int64_t)idxs[i] : ((v.n_frames == 1) ? 0 : i);
    T *fo = out + f * v.D * v.H * v.W;
    walk3(L, (int)(u & 3), flags, [&](const int64_t *p, T err) {
        if (!(err <= T(1)) || p[0] < 0 || p[0] >= v.W || p[1] < 0 || p[1] >= v.H || p[2] < 0 || p[2] >= v.D) return;
        apply_atomic<OV>(fo + (p[2] * v.H + p[1]) * v.W + p[0], pixel_value<K>(err, max_val));
    });
}

// Two-phase draw: planes of every line recorded by one lane per line
// (k_walk3_main), then one lane per (plane, quadrant) fills (k_fill3), so the
// lanes of a wave run consecutive planes of one line, whose fills take about
// as many steps each (one lane per line left most of a wave idle behind its
// longest and widest line).

//
// The walk is a serial chain, so its time is the instructions of a step times the
// longest line.  One loop for all long axes (walk3_main's, unrolled for each, left
// a wave of mixed lines running three in turn), increments known before it, moves
// by selects: 50 000 lines of up to 40 voxels 72 -> 29 us.
template <typename T>
__global__ void __launch_bounds__(D3_NT)
k_walk3_main(const T *__restrict__ lines, int64_t n_lines, const int64_t *__restrict__ off,
             PlaneState<T> *__restrict__ states, int *__restrict__ flags)
{
    const int64_t i = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (i >= n_lines) return;
    const int64_t base = off[i], cap = off[i + 1] - base;
    if (cap == 0) return;
    PlaneState<T> *const dst = states + base;
    const int most = (int)min(cap, (int64_t)INT_MAX);
    int k = 0;
    Line3<T> L;
    if (line3_setup(lines + 7 * i, L) == 1) {
        Iter3<T> it;
        it3_start(L, it);
        const int s0 = (int)L.step[0], s1 = (int)L.step[1], s2 = (int)L.step[2];
        const T t0 = (T)s0 * L.t[0], t1 = (T)s1 * L.t[1], t2 = (T)s2 * L.t[2];
        // the normal errors' changes: pair (0,1) along 0, 1; (0,2) along 0, 2; (1,2) along 1, 2
        const T a0 = (T)s0 * L.nrm[0][0], a1 = (T)s1 * L.nrm[0][1], b0 = (T)s0 * L.nrm[1][0], b2 = (T)s2 * L.nrm[1][2],
                c1 = (T)s1 * L.nrm[2][1], c2 = (T)s2 * L.nrm[2][2];
        // steps to the walk's end along each axis, and the budget of all of them
        int l0 = (int)((L.m1[0] - L.m0[0]) * s0), l1 = (int)((L.m1[1] - L.m0[1]) * s1),
            l2 = (int)((L.m1[2] - L.m0[2]) * s2);
        int64_t budget = (int64_t)l0 + l1 + l2 + 64;
        T te = it.te, na = it.ne[0], nb = it.ne[1], nc = it.ne[2];
        int x = (int)it.cur[0], y = (int)it.cur[1], z = (int)it.cur[2];
        // a pair's choice (it3_update): whether its first and second axis may step
        auto choice = [](T n, T u, T v, bool &first, bool &second) {
            const T ex = n + u, ey = n + v, exy = ex + v;
            const bool q = m_abs(ey) < m_abs(ex);
            const bool both = m_abs(exy) < m_abs(q ? ey : ex);
            first = !q | both;
            second = q | both;
        };
        bool go = (l0 != 0) & (l1 != 0) & (l2 != 0);
        while (go) {
            bool a_0, a_1, b_0, b_2, c_1, c_2;
            choice(na, a0, a1, a_0, a_1);
            choice(nb, b0, b2, b_0, b_2);
            choice(nc, c1, c2, c_1, c_2);
            const bool m0 = a_0 & b_0, m1 = a_1 & c_1, m2 = b_2 & c_2;
            if ((L.axis == 0) ? m0 : ((L.axis == 1) ? m1 : m2)) {
                if (k == most) {   // cannot happen: one plane per long-axis step
                    atomicOr(flags, FLAG_STUCK);
                    break;
                }
                PlaneState<T> ps;
                ps.te = te;
                ps.ne[0] = na;
                ps.ne[1] = nb;
                ps.ne[2] = nc;
                ps.cur[0] = x;
                ps.cur[1] = y;
                ps.cur[2] = z;
                ps.line = (int32_t)i;
                dst[k++] = ps;
            }
            if (budget-- == 0) {
                atomicOr(flags, FLAG_STUCK);
                break;
            }
            te += m0 ? t0 : T(0);
            te += m1 ? t1 : T(0);
            te += m2 ? t2 : T(0);
            na += m0 ? a0 : T(0);
            na += m1 ? a1 : T(0);
            nb += m0 ? b0 : T(0);
            nb += m2 ? b2 : T(0);
            nc += m1 ? c1 : T(0);
            nc += m2 ? c2 : T(0);
            x += m0 ? s0 : 0;
            y += m1 ? s1 : 0;
            z += m2 ? s2 : 0;
            l0 -= m0 ? 1 : 0;
            l1 -= m1 ? 1 : 0;
            l2 -= m2 ? 1 : 0;
            go = (l0 != 0) & (l1 != 0) & (l2 != 0);
        }
    }
    for (int64_t q = k; q < cap; q++) dst[q].line = -1;
}

// A line's constants for the fills of its planes: Line3's, and what turns their
// divisions into products (a correctly rounded reciprocal and one correction
// step give the IEEE quotient).
template <typename T>
struct alignas(16) Rec3 {
    T t[3];              // p1 - p0: the pair normals are (t[b], -t[a])
    T len, rlen, LL, w2;
    T in, out;           // sum of the squared normal errors, times len^2: below `in` the pixel is within w, above `out` beyond
    double rw2;          // 1 / (double)w2
    int64_t frame;
    int32_t ray_cap;
    int32_t span[3];     // steps a plane's pixels lie from its centre along each axis (patch size: a few may lie further)
    int8_t axis, step[3];
};

__device__ __forceinline__ float div3(float a, float b, float rb) { return div_rn(a, b, rb); }
__device__ __forceinline__ double div3(double a, double b, double rb) { return div_rn(a, b, rb); }

// it3_nerr with the reciprocal: the square of a float is exact in double, so one
// FMA rounds like the reference's double addition
__device__ __forceinline__ float nerr3(const Rec3<float> &L, const float *ne)
{
    float e = 0.0f;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double v = (double)div3(ne[q], L.len, L.rlen);
        e = (float)__builtin_fma(v, v, (double)e);
    }
    return e;
}

__device__ __forceinline__ double nerr3(const Rec3<double> &L, const double *ne)
{
    double e = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double v = div3(ne[q], L.len, L.rlen);
        e = e + v * v;
    }
    return e;
}

__device__ __forceinline__ float err3(const Rec3<float> &L, float te, float nerr)
{
    const float a = -te, b = te - L.LL, m = (a < b) ? b : a, at = (m < 0.0f) ? 0.0f : m;
    const double qt = (double)div3(at, L.len, L.rlen);
    return (float)div_rn(__builtin_fma(qt, qt, (double)nerr), (double)L.w2, L.rw2);
}

__device__ __forceinline__ double err3(const Rec3<double> &L, double te, double nerr)
{
    const double a = -te, b = te - L.LL, m = (a < b) ? b : a, at = (m < 0.0) ? 0.0 : m;
    const double qt = div3(at, L.len, L.rlen), qt2 = qt * qt;
    return (qt2 + nerr) / L.w2;
}

// Validation (as k_check3), ub[i]: planes of line i at most (the long-axis span),
// 0 if it draws nothing (ub[n_lines] = 0: the scan's total), and its record.
template <typename T, typename I>
__global__ void __launch_bounds__(D3_NT)
k_setup3(const T *__restrict__ lines, int64_t n_lines, const I *__restrict__ idxs, Vol3 v, int *__restrict__ flags,
         int64_t *__restrict__ ub, Rec3<T> *__restrict__ rec)
{
    const int64_t i = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (i > n_lines) return;
    int64_t n = 0;
    if (i < n_lines) {
        const int64_t f = idxs ? (int64_t)idxs[i] : ((v.n_frames == 1) ? 0 : i);
        if (f < 0 || f >= v.n_frames) atomicOr(flags, FLAG_INDEX);
        Line3<T> L;
        const int rc = line3_setup(lines + 7 * i, L);
        if (rc < 0) atomicOr(flags, FLAG_LONG);
        if (rc == 1) {
            const int a = L.axis;
            const int64_t m0 = (a == 0) ? L.m0[0] : ((a == 1) ? L.m0[1] : L.m0[2]);
            const int64_t m1 = (a == 0) ? L.m1[0] : ((a == 1) ? L.m1[1] : L.m1[2]);
            n = (m1 > m0) ? m1 - m0 : m0 - m1;
            Rec3<T> R;
            for (int k = 0; k < 3; k++) {
                R.t[k] = L.t[k];
                R.step[k] = (int8_t)L.step[k];
            }
            R.len = L.len;
            R.rlen = T(1) / L.len;
            R.LL = L.len * L.len;
            R.w2 = L.w2;
            R.rw2 = 1.0 / (double)L.w2;
            const double lim = (double)L.w2 * (double)L.len * (double)L.len, tol = sizeof(T) == 4 ? 4e-6 : 1e-13;
            R.in = (T)(lim * (1.0 - tol));
            R.out = (T)(lim * (1.0 + tol));
            // Squares near the smallest normal number are not accurate to tol, nor is the
            // correction of a quotient: the limits decide nothing then, and a reciprocal of 0
            // makes div_rn divide.
            if (!(lim > (sizeof(T) == 4 ? 1e-30 : 1e-290))) {
                R.rlen = T(0);
                R.in = T(0);
                R.out = (T)__builtin_inf();
            }
            const T ta = (a == 0) ? L.t[0] : ((a == 1) ? L.t[1] : L.t[2]);
            for (int k = 0; k < 3; k++) {
                const float slope = (float)(L.t[k] / ta);
                R.span[k] = (int32_t)fminf((float)lines[7 * i + 6] * sqrtf(1.0f + slope * slope) + 0.5f, 1e6f);
            }
            R.frame = f;
            R.ray_cap = (int32_t)min(L.ray_cap, (int64_t)INT_MAX);
            R.axis = (int8_t)a;
            rec[i] = R;
        }
    }
    ub[i] = n;
}

__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t patch_bits(float v) { return __float_as_uint(v); }
__device__ __forceinline__ unsigned long long patch_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
__device__ __forceinline__ float patch_value(uint32_t b) { return __uint_as_float(b); }
__device__ __forceinline__ double patch_value(unsigned long long b) { return __longlong_as_double((long long)b); }

// Fills of the recorded planes.  A wave takes 2^planes_log consecutive planes, one
// (plane, quadrant) per lane (fill3_quadrant's pixels: a walk away from the
// line with, from each of its pixels, a ray along the other axis for each axis
// that the next step moves).  Walk and rays are one loop, a candidate pixel of
// every lane per turn, written in terms of the plane's axes P < Q, so that
// lanes at different places of their walks and on different axes stay
// together; the pixels inside go to the wave's queue, whose errors and profile
// values 64 lanes compute at a time.
//
// The volume is updated with global atomics, whose rate is one request per 64
// bytes and instruction: 13 M float additions take 621 us at random places, 189
// us in runs of 4 along x, 81 us in runs of 16.  So the values of a plane
// across y or z first go to a patch of the plane in LDS, whose rows along x are
// then added by neighbouring lanes; planes across x (their pixels at one place
// of consecutive planes are neighbours in x, and in the queue) and pixels
// outside the patch are added directly.
//
// Bound by the loop's vector instructions (191 M wave instructions, 310 us at
// the issue rate, for 50 000 lines of widths 1 to 3, 13 M voxels, in 16 volumes
// of 64 x 128 x 128).  A wave's patch and queue limit the waves in flight: with
// patches of 1536, 1024, 768, 640 values 526, 433, 387, 381 us (planes that
// find no room in the patch are added directly, so not smaller still).  Planes
// whose rows reach less than 2 steps from the centre have too few neighbours to
// gather: 200 000 lines of widths 0.2 to 0.6 take 396 us with patches, 283 without
// (349 with one lane per (plane, quadrant)).
// For max hardly any voxel is written (most are below what is there), so its
// patch is kept to the smallest planes: 525 us with the patches of the sums, 465
// with 64 values; 20 000 lines of widths 2 to 6 in doubles 984 and 795.
// One lane per (plane, quadrant) with atomics for every pixel took 623 us.
constexpr int FILL_PLANES = 16, FILL_NT = 256, FILL_QUEUE = 128;

//
// RAYS: for so few planes that the widest one's quadrant, its lane's chain of steps, is
// the time.  While every lane of the wave is on a ray, its steps run in a loop of their
// own (a third of the instructions): 50 lines of widths 10 to 25 743 -> 504 us.  With
// full waves that seldom happens, and the second copy of the loop costs (50 000 lines
// 423 -> 460).  One instance for all profiles (K_MIXED, the profile in kid).
template <typename T, int K, int OV, bool RAYS>
__global__ void __launch_bounds__(FILL_NT)
k_fill3(T *__restrict__ out, const Rec3<T> *__restrict__ rec, const PlaneState<T> *__restrict__ states,
        int64_t n_states, int planes_log, Vol3 v, T max_val, int kid, int *__restrict__ flags)
{
    constexpr int NW = FILL_NT / 64, PATCH = (OV == 1) ? 64 : (sizeof(T) == 4 ? 768 : 512);
    using Bits = typename std::conditional<sizeof(T) == 4, uint32_t, unsigned long long>::type;
    struct Entry {   // a pixel to draw: its errors, its plane (4 bits) and offsets from the centre along P, Q (14 bits each)
        T te, ne[3];
        uint32_t at;
    };
    struct Plane {
        int64_t centre;   // index of its centre in `out`
        int32_t line, patch, spanP, spanQ;
        int32_t sP, sQ;   // strides along P, Q
    };
    __shared__ Entry queue[NW][FILL_QUEUE];
    __shared__ Bits patch[NW][PATCH];
    __shared__ Plane plane[NW][FILL_PLANES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t below = (1ull << lane) - 1ull;
    const int planes = 1 << planes_log;
    const int64_t first = ((int64_t)blockIdx.x * NW + wave) << planes_log;
    const int pl = lane & (planes - 1), quad = lane >> planes_log;
    const bool have = quad < 4 && first + pl < n_states;
    PlaneState<T> ps;
    ps.line = -1;
    if (have) ps = states[first + pl];
    bool go = ps.line >= 0;

    T te = T(0), ne[3], xte = T(0), xne[3], s_in = T(0), s_out = T(0), stP = T(0), stQ = T(0);
    T iP[3], iQ[3];   // changes of the three normal errors per step along P, Q (one of them zero each)
    int count = 0, walks = 0, cap = 0, plane_q = 0;   // count, walks: steps of the ray, of the walk
    // offsets from the centre along P, Q (of the candidate, of the walk), steps, offsets inside the volume
    int oP = 0, oQ = 0, xP = 0, xQ = 0, dP = 0, dQ = 0, loP = 0, hiP = -1, loQ = 0, hiQ = -1, side = 0;
    bool second = false, alongP = false, flat = false;
    const Rec3<T> *L = rec;
    for (int k = 0; k < 3; k++) ne[k] = xne[k] = iP[k] = iQ[k] = T(0);
    if (go) {
        L = rec + ps.line;
        const int a = L->axis;
        const int P = (a == 0) ? 1 : 0, Q = (a == 2) ? 1 : 2;
        const T t0 = L->t[0], t1 = L->t[1], t2 = L->t[2];
        const T tP = (P == 0) ? t0 : t1, tQ = (Q == 1) ? t1 : t2;
        const bool flip1 = quad & 1, flip2 = quad >> 1;   // of axes (a + 1) % 3, (a + 2) % 3
        dP = ((P == 0) ? L->step[0] : L->step[1]) * (((a == 1) ? flip2 : flip1) ? -1 : 1);
        dQ = ((Q == 1) ? L->step[1] : L->step[2]) * (((a == 1) ? flip1 : flip2) ? -1 : 1);
        const T fP = (T)dP, fQ = (T)dQ;
        stP = fP * tP;
        stQ = fQ * tQ;
        // pairs (0,1), (0,2), (1,2): normals (t[b], -t[a])
        iP[0] = fP * ((P == 0) ? t1 : -t0);
        iP[1] = (P == 0) ? fP * t2 : T(0);
        iP[2] = (P == 0) ? T(0) : fP * t2;
        iQ[0] = (Q == 1) ? fQ * -t0 : T(0);
        iQ[1] = (Q == 1) ? T(0) : fQ * -t0;
        iQ[2] = (Q == 1) ? fQ * t2 : fQ * -t1;
        plane_q = (a == 0) ? 2 : ((a == 1) ? 1 : 0);
        s_in = L->in;
        s_out = L->out;
        cap = L->ray_cap;
        const int64_t ca = (a == 0) ? ps.cur[0] : ((a == 1) ? ps.cur[1] : ps.cur[2]);
        const int64_t da = (a == 0) ? v.W : ((a == 1) ? v.H : v.D);
        const int cP = (P == 0) ? ps.cur[0] : ps.cur[1], cQ = (Q == 1) ? ps.cur[1] : ps.cur[2];
        const int64_t nP = (P == 0) ? v.W : v.H, nQ = (Q == 1) ? v.H : v.D;
        const int64_t strP = (P == 0) ? 1 : v.W, strQ = (Q == 1) ? v.W : v.W * v.H;
        // offsets inside the volume (MAX_VISITS3 keeps a plane's pixels well within 2^13 of its centre: Entry::at);
        // a plane outside of it draws nothing
        flat = ca >= 0 && ca < da;
        loP = (int)max(-(int64_t)cP, (int64_t)-8191);
        hiP = (int)min(nP - 1 - cP, (int64_t)8191);
        loQ = (int)max(-(int64_t)cQ, (int64_t)-8191);
        hiQ = (int)min(nQ - 1 - cQ, (int64_t)8191);
        if (!flat) hiP = loP - 1;
        te = ps.te;
        for (int k = 0; k < 3; k++) ne[k] = ps.ne[k];
        const bool one = flip1 != flip2;   // the first step: along (a + 2) % 3 when exactly one axis is flipped
        alongP = (a == 1) ? one : !one;
        const int spanP = (P == 0) ? L->span[0] : L->span[1], spanQ = (Q == 1) ? L->span[1] : L->span[2];
        side = (a != 0 && flat && spanP >= 2 && spanP < 32 && spanQ < 32) ? (2 * spanP + 1) * (2 * spanQ + 1) : 0;
        if (quad == 0) {
            Plane &p = plane[wave][pl];
            p.centre = ((L->frame * v.D + ps.cur[2]) * v.H + ps.cur[1]) * v.W + ps.cur[0];
            p.line = ps.line;
            p.spanP = spanP;
            p.spanQ = spanQ;
            p.sP = (int32_t)strP;
            p.sQ = (int32_t)strQ;
        }
    }
    // patches one after the other (a plane whose patch does not fit has none)
    {
        int x = side;
#pragma unroll
        for (int d = 1; d < FILL_PLANES; d <<= 1) {
            const int y = __shfl_up(x, d, 64);   // (a quadrant's lanes are neighbours)
            if (pl >= d) x += y;
        }
        if (quad == 0) plane[wave][pl].patch = (side > 0 && x <= PATCH) ? x - side : -1;
        const int all = min(__shfl(x, planes - 1, 64), PATCH);
        for (int i = lane; i < all; i += 64) patch[wave][i] = (Bits)~(Bits)0;   // (a NaN that no value has)
    }
    wave_fence();
    auto put = [&](T pte, const T *pne, uint32_t at) {
        const Plane &p = plane[wave][at >> 28];
        const int qP = (int)((at >> 14) & 0x3fffu) - 8192, qQ = (int)(at & 0x3fffu) - 8192;
        const bool held = p.patch >= 0 && abs(qP) <= p.spanP && abs(qQ) <= p.spanQ;
        const auto voxel = [&]() { return out + (p.centre + (int64_t)qP * p.sP + (int64_t)qQ * p.sQ); };
        // (the voxel is inside the volume; its value arrives while the new one is computed)
        T now = T(0);
        if (OV == 1 && !held) now = value_now(voxel());
        const Rec3<T> &R = rec[p.line];
        const T e = err3(R, pte, nerr3(R, pne));
        if (!(e <= T(1))) return;
        const T val = pixel_value_of<K>(kid, e, max_val);
        if (held)
            patch[wave][p.patch + (qQ + p.spanQ) * (2 * p.spanP + 1) + qP + p.spanP] = patch_bits(val);
        else
            apply_atomic<OV>(voxel(), val, now);
    };
    int q_head = 0, q_tail = 0;   // the wave's queue (uniform over the wave)
    auto drain = [&](int n) {
        wave_fence();
        if (lane < n) {
            const Entry e = queue[wave][(q_head + lane) & (FILL_QUEUE - 1)];
            put(e.te, e.ne, e.at);
        }
        q_head += n;
        wave_fence();
    };
    auto push = [&](bool mine) {
        const uint64_t m = __ballot(mine);
        if (m == 0) return;
        if (mine) {
            Entry &e = queue[wave][(q_tail + __popcll(m & below)) & (FILL_QUEUE - 1)];
            e.te = te;
            for (int k = 0; k < 3; k++) e.ne[k] = ne[k];
            e.at = ((uint32_t)pl << 28) | ((uint32_t)(oP + 8192) << 14) | (uint32_t)(oQ + 8192);
        }
        q_tail += __popcll(m);
        if (q_tail - q_head >= 64) drain(64);
    };
    // the plane's centre, without the band test
    push(go && quad == 0 && loP <= 0 && hiP >= 0 && loQ <= 0 && hiQ >= 0);
    // the quadrant's first pixel
    te += alongP ? stP : stQ;
    for (int k = 0; k < 3; k++) ne[k] += alongP ? iP[k] : iQ[k];
    oP = alongP ? dP : 0;
    oQ = alongP ? 0 : dQ;
    int dir = 0;           // 0: the walk's own pixel, 1: a ray along Q, 2: a ray along P
    bool nP = false, nQ = false;
    while (__ballot(go)) {
        const T s2 = ne[0] * ne[0] + ne[1] * ne[1] + ne[2] * ne[2];
        bool in = go && s2 < s_in;
        if (go && !in && !(s2 > s_out)) in = nerr3(*L, ne) < L->w2;
        if (in && (count == cap || walks == cap)) {
            atomicOr(flags, FLAG_STUCK);
            go = in = false;
        }
        push(in && oP >= loP && oP <= hiP && oQ >= loQ && oQ <= hiQ);
        // the next candidate: from the pixel before or from the walk's
        const bool walk = dir == 0;
        go = go && (in || !walk);
        if (walk) {
            // the walk's pixel: keep it, and its next step (it3_update)
            xte = te;
            for (int k = 0; k < 3; k++) xne[k] = ne[k];
            xP = oP;
            xQ = oQ;
            const T w = (plane_q == 0) ? ne[0] : ((plane_q == 1) ? ne[1] : ne[2]);
            const T gP = (plane_q == 0) ? iP[0] : ((plane_q == 1) ? iP[1] : iP[2]);
            const T gQ = (plane_q == 0) ? iQ[0] : ((plane_q == 1) ? iQ[1] : iQ[2]);
            const T eP = w + gP, eQ = w + gQ, eb = eP + gQ;
            const bool qb = m_abs(eQ) < m_abs(eP);
            const bool both = m_abs(eb) < m_abs(qb ? eQ : eP);
            nP = !qb || both;
            nQ = qb || both;
        }
        const bool on = in && !walk;                 // the ray goes on
        second = !in && dir == 1 && nQ;              // the ray along P comes next
        const bool step = !walk && !in && !second;   // the walk's next step
        const bool mP = on ? dir == 2 : (walk ? !nP : (second || nP));
        const bool mQ = on ? dir == 1 : (walk ? nP : (!second && nQ));
        count = on ? count + 1 : 0;
        walks += step ? 1 : 0;
        te = on ? te : xte;
        te += mP ? stP : T(0);
        te += mQ ? stQ : T(0);
        for (int k = 0; k < 3; k++) {
            ne[k] = on ? ne[k] : xne[k];
            ne[k] += mP ? iP[k] : T(0);
            ne[k] += mQ ? iQ[k] : T(0);
        }
        oP = (on ? oP : xP) + (mP ? dP : 0);
        oQ = (on ? oQ : xQ) + (mQ ? dQ : 0);
        dir = on ? dir : (walk ? (nP ? 1 : 2) : (second ? 2 : 0));
        if constexpr (RAYS) {
            if (__ballot(go && !on) != 0) continue;
            const bool rP = dir == 2;
            const T st = rP ? stP : stQ, i0 = rP ? iP[0] : iQ[0], i1 = rP ? iP[1] : iQ[1], i2 = rP ? iP[2] : iQ[2];
            const int sP = rP ? dP : 0, sQ = rP ? 0 : dQ;
            while (__ballot(go)) {
                const T r2 = ne[0] * ne[0] + ne[1] * ne[1] + ne[2] * ne[2];
                if (__ballot(go && !(r2 < s_in && count < cap)) != 0) break;   // (for the step above)
                push(go && oP >= loP && oP <= hiP && oQ >= loQ && oQ <= hiQ);
                count++;
                te += st;
                ne[0] += i0;
                ne[1] += i1;
                ne[2] += i2;
                oP += sP;
                oQ += sQ;
            }
        }
    }
    drain(q_tail - q_head);
    // the patches' rows
    for (int k = 0; k < planes; k++) {
        if (first + k >= n_states) break;
        const bool used = __shfl(side, k, 64) > 0;
        if (!used) continue;
        const Plane &p = plane[wave][k];
        if (p.patch < 0) continue;
        const int n = 2 * p.spanP + 1, all = n * (2 * p.spanQ + 1);
        const float rn = 1.0f / (float)n;
        T *const o = out + p.centre;
        for (int i = lane; i < all; i += 64) {
            const Bits bits = patch[wave][p.patch + i];
            if (bits == (Bits)~(Bits)0) continue;
            const int y = (int)(((float)i + 0.5f) * rn), x = i - y * n;
            apply_atomic<OV>(o + ((int64_t)(x - p.spanP) * p.sP + (int64_t)(y - p.spanQ) * p.sQ), patch_value(bits));
        }
    }
}

// accumulate_lines, mixed overlaps: the lines of terms [t0, t0 + nb) drawn
// into their term's zeroed buffer with in_overlap (the reference's term
// buffer: 0 + v, or std::max(0, v) from zero),
// every drawn voxel marked in `touched`
template <typename T, typename I, int K, int IN_OV>
__global__ void __launch_bounds__(D3_NT)
k_acc3_draw(T *__restrict__ buf, uint32_t *__restrict__ touched, const T *__restrict__ lines, int64_t n_lines,
            const I *__restrict__ terms, int64_t t0, int64_t nb, Vol3 v, T max_val, int *__restrict__ flags)
{
    const int64_t u = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (u >= 4 * n_lines) return;
    const int64_t i = u >> 2;
    const int64_t b = (int64_t)terms[i] - t0;
    if (b < 0 || b >= nb) return;
    Line3<T> L;
    if (line3_setup(lines + 7 * i, L) != 1) return;
    const int64_t V = v.D * v.H * v.W;
    walk3(L, (int)(u & 3), flags, [&](const int64_t *p, T err) {
        if (!(err <= T(1)) || p[0] < 0 || p[0] >= v.W || p[1] < 0 || p[1] >= v.H || p[2] < 0 || p[2] >= v.D) return;
        const int64_t k = b * V + (p[2] * v.H + p[1]) * v.W + p[0];
        apply_atomic<IN_OV>(buf + k, pixel_value<K>(err, max_val));
        atomicOr(&touched[k >> 5], 1u << (k & 31));
    });
}

// every touched voxel of the batch combined into frame frames[term] with
// out_overlap (buffer + out, or std::max(out, buffer)); buffer and marks reset
template <typename T, typename I, int OUT_OV>
__global__ void __launch_bounds__(D3_NT)
k_acc3_fold(T *__restrict__ out, T *__restrict__ buf, uint32_t *__restrict__ touched, const I *__restrict__ frames,
            int64_t t0, int64_t nb, Vol3 v)
{
    const int64_t V = v.D * v.H * v.W;
    const int64_t k = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (k >= nb * V) return;
    const uint32_t bit = 1u << (k & 31);
    if (!(touched[k >> 5] & bit)) return;
    const int64_t b = k / V, r = k - b * V;
    apply_atomic<OUT_OV>(out + (int64_t)frames[t0 + b] * V + r, buf[k]);
    buf[k] = T(0);
}

__global__ void k_clear_words(uint32_t *__restrict__ w, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (i < n) w[i] = 0u;
}

// frame of every line (frames[terms[i]]) and the range checks of
// accumulate_lines (bresenham.cpp:171-187)
template <typename I>
__global__ void __launch_bounds__(D3_NT)
k_term_frames3(const I *__restrict__ terms, const I *__restrict__ frames, int64_t n_lines, int64_t n_terms,
               int64_t n_frames, I *__restrict__ comp, int *__restrict__ bad)
{
    const int64_t i = (int64_t)blockIdx.x * D3_NT + threadIdx.x;
    if (i < n_terms && (frames[i] < 0 || (int64_t)frames[i] >= n_frames)) atomicOr(&bad[1], 1);
    if (i >= n_lines) return;
    const I t = terms[i];
    if (t < 0 || (int64_t)t >= n_terms) {
        atomicOr(&bad[0], 1);
        return;
    }
    if (comp) comp[i] = frames[t];
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
static int check_vol(int64_t n_frames, int64_t D, int64_t H, int64_t W, int64_t n_lines, int kernel, int overlap)
{
    if (n_frames < 0 || D < 0 || H < 0 || W < 0 || n_lines < 0) return fail(CBX_EVALUE, "negative size");
    if (n_lines >= (int64_t(1) << 34)) return fail(CBX_EVALUE, "too many lines");
    if (kernel < 0 || kernel > 4) return fail(CBX_EVALUE, "kernel is missing");
    if (overlap < 0 || overlap > 1) return fail(CBX_EVALUE, "Invalid overlap keyword");
    return CBX_OK;
}

static int read_flags(const int *flags, hipStream_t st, int *hv)
{
    uint64_t v = 0;
    const void *src[1] = {flags};
    const int bytes[1] = {4};
    CBX_HIP(read_device_values(st, 1, src, bytes, &v));
    *hv = (int)v;
    return CBX_OK;
}

static int flags3_status(int hv)
{
    if (hv & FLAG_INDEX) return fail(CBX_EINDEX, "idxs is outside of (0, n_frames)");
    if (hv & FLAG_LONG)
        return fail(CBX_EVALUE, "a line's 3D walk exceeds the supported length (2^26 px), coordinate range (1e9) "
                                "or pixel count (2^30)");
    if (hv & FLAG_STUCK) return fail(CBX_ERUNTIME, "a line walk did not terminate within its step budget");
    return CBX_OK;
}

// every line checked before anything is drawn; flags left zeroed for the draw
template <typename T, typename I>
static int validate3(const T *lines, int64_t n_lines, const I *idxs, const Vol3 &v, int *flags, hipStream_t st)
{
    CBX_HIP(hipMemsetAsync(flags, 0, sizeof(int), st));
    k_check3<T, I><<<grid_for(n_lines, D3_NT), D3_NT, 0, st>>>(lines, n_lines, idxs, v, flags);
    CBX_HIP(hipGetLastError());
    int hv = 0, rc = read_flags(flags, st, &hv);
    return rc ? rc : flags3_status(hv);
}

template <typename T, typename I, int OV>
static void launch_draw3(int kernel, T *out, const T *lines, int64_t n, const I *idxs, const Vol3 &v, T mv,
                         int *flags, hipStream_t st)
{
    const unsigned g = (unsigned)grid_for(4 * n, D3_NT);   // four lanes per line
    switch (kernel) {
    case K_BIWEIGHT: k_draw3<T, I, K_BIWEIGHT, OV><<<g, D3_NT, 0, st>>>(out, lines, n, idxs, v, mv, flags); break;
    case K_GAUSSIAN: k_draw3<T, I, K_GAUSSIAN, OV><<<g, D3_NT, 0, st>>>(out, lines, n, idxs, v, mv, flags); break;
    case K_PARABOLIC: k_draw3<T, I, K_PARABOLIC, OV><<<g, D3_NT, 0, st>>>(out, lines, n, idxs, v, mv, flags); break;
    case K_RECTANGULAR:
        k_draw3<T, I, K_RECTANGULAR, OV><<<g, D3_NT, 0, st>>>(out, lines, n, idxs, v, mv, flags);
        break;
    default: k_draw3<T, I, K_TRIANGULAR, OV><<<g, D3_NT, 0, st>>>(out, lines, n, idxs, v, mv, flags); break;
    }
}

template <typename T, int OV>
static void launch_fill3(int kernel, T *out, const Rec3<T> *rec, const PlaneState<T> *states, int64_t n_states,
                         const Vol3 &v, T mv, int *flags, hipStream_t st)
{
    // Planes of a wave: 16, or fewer where that would leave SIMDs without a wave to
    // work for the widest planes (us with 16 / 8 / 4 / 2 planes: 62 000 planes of widths 5 to
    // 9 397 / 353 / 352 / 514, 15 000 of 10 to 25 1133 / 855 / 700 / 862, 3800 of them 1257 /
    // 966 / 817 / 741, with RAYS and one 504; 2.8 M of 0.2 to 0.6 283 / 412 / 648 / 1100).
    const bool rays = n_states < 8192;
    const int planes_log = rays ? 0 : (n_states < 32768 ? 2 : (n_states < 131072 ? 3 : 4));
    const int64_t per_group = (int64_t)(FILL_NT / 64) << planes_log;
    const unsigned g = (unsigned)((n_states + per_group - 1) / per_group);
#define CBX_FILL3(KK, RAYS)                                                                                     \
    k_fill3<T, KK, OV, RAYS><<<g, FILL_NT, 0, st>>>(out, rec, states, n_states, planes_log, v, mv, kernel, flags)
    if (rays) {
        CBX_FILL3(K_MIXED, true);
        return;
    }
    switch (kernel) {
    case K_BIWEIGHT: CBX_FILL3(K_BIWEIGHT, false); break;
    case K_GAUSSIAN: CBX_FILL3(K_GAUSSIAN, false); break;
    case K_PARABOLIC: CBX_FILL3(K_PARABOLIC, false); break;
    case K_RECTANGULAR: CBX_FILL3(K_RECTANGULAR, false); break;
    default: CBX_FILL3(K_TRIANGULAR, false); break;
    }
#undef CBX_FILL3
}

// validation, the draw, then its step-budget flag (inside an open Workspace).
// Above MAX_PLANES recorded planes, or with strides or widths that the fills'
// 32-bit offsets do not hold, the single-kernel walk (four lanes per line)
// runs instead of the two phases.
template <typename T, typename I>
static int draw3_run(T *out, const Vol3 &v, const T *lines, int64_t n_lines, const I *idxs, T max_val, int kernel,
                     int overlap, hipStream_t st)
{
    DevBuf<int> flags;
    DevBuf<int64_t> ub, off;
    DevBuf<Rec3<T>> rec;
    CBX_HIP(flags.alloc(1, st));
    CBX_HIP(ub.alloc((size_t)n_lines + 1, st));
    CBX_HIP(off.alloc((size_t)n_lines + 1, st));
    CBX_HIP(rec.alloc((size_t)n_lines, st));
    {
        void *const zp[1] = {flags.ptr};
        const int64_t zw[1] = {1};
        CBX_HIP(zero_words(st, 1, zp, zw));
    }
    // checks, records and the planes of every line: offsets by a scan of their bounds
    k_setup3<T, I><<<grid_for(n_lines + 1, D3_NT), D3_NT, 0, st>>>(lines, n_lines, idxs, v, flags.ptr, ub.ptr, rec.ptr);
    CBX_HIP(hipGetLastError());
    CBX_HIP(exclusive_scan_i64(ub.ptr, off.ptr, n_lines + 1, st));
    uint64_t total = 0;
    int rc;
    {
        uint64_t hv[2];
        const void *src[2] = {off.ptr + n_lines, flags.ptr};
        const int nb[2] = {8, 4};
        CBX_HIP(read_device_values(st, 2, src, nb, hv));
        total = hv[0];
        if ((rc = flags3_status((int)hv[1]))) return rc;
    }
    if (max_val != max_val) max_val = (T)NAN;   // (k_fill3's patches keep one pattern for themselves)
    DevBuf<PlaneState<T>> states;
    const bool two_phase = total <= (uint64_t)MAX_PLANES && v.W * v.H < (int64_t(1) << 31) && n_lines < INT_MAX;
    if (two_phase && total > 0) CBX_HIP(states.alloc((size_t)total, st));
    {
        KernelTimer timer("draw3", st);
        if (two_phase) {
            if (total > 0) {
                k_walk3_main<T><<<grid_for(n_lines, D3_NT), D3_NT, 0, st>>>(lines, n_lines, off.ptr, states.ptr,
                                                                           flags.ptr);
                if (overlap == 0)
                    launch_fill3<T, 0>(kernel, out, rec.ptr, states.ptr, (int64_t)total, v, max_val, flags.ptr, st);
                else
                    launch_fill3<T, 1>(kernel, out, rec.ptr, states.ptr, (int64_t)total, v, max_val, flags.ptr, st);
            }
        } else if (overlap == 0) {
            launch_draw3<T, I, 0>(kernel, out, lines, n_lines, idxs, v, max_val, flags.ptr, st);
        } else {
            launch_draw3<T, I, 1>(kernel, out, lines, n_lines, idxs, v, max_val, flags.ptr, st);
        }
        CBX_HIP(hipGetLastError());
    }
    int hv = 0;
    if ((rc = read_flags(flags.ptr, st, &hv))) return rc;
    return flags3_status(hv);
}

template <typename T, typename I>
static int draw_lines3(T *out, int64_t n_frames, int64_t D, int64_t H, int64_t W, const T *lines, int64_t n_lines,
                       const I *idxs, T max_val, int kernel, int overlap, void *stream)
{
    int rc = check_vol(n_frames, D, H, W, n_lines, kernel, overlap);
    if (rc) return rc;
    // idxs = None: one frame, or one frame per line (bresenham.cpp:5-20)
    if (!idxs && n_lines > 0 && n_frames != 1 && n_frames != n_lines)
        return fail(CBX_EVALUE, "idxs has an incompatible size (" + std::to_string(n_lines) + " != " +
                                    std::to_string(n_frames) + ")");
    if (n_lines == 0 || n_frames * D * H * W == 0) return CBX_OK;
    hipStream_t st = (hipStream_t)stream;
    Workspace ws(st);
    return draw3_run(out, Vol3{n_frames, D, H, W}, lines, n_lines, idxs, max_val, kernel, overlap, st);
}

// mixed overlaps: terms in batches of at most 256 MiB of term buffers
template <typename T, typename I, int K, int IN_OV, int OUT_OV>
static int accumulate3_batches(T *out, const T *lines, int64_t n_lines, const I *terms, const I *frames,
                               int64_t n_terms, const Vol3 &v, T max_val, int *flags, hipStream_t st)
{
    const int64_t V = v.D * v.H * v.W;
    const int64_t budget = int64_t(256) << 20;
    const int64_t nb = std::max<int64_t>(1, std::min<int64_t>(n_terms, budget / (V * (int64_t)sizeof(T))));
    const int64_t words = (nb * V + 31) / 32;
    DevBuf<T> buf;
    DevBuf<uint32_t> touched;
    CBX_HIP(buf.alloc((size_t)(nb * V), st));
    CBX_HIP(touched.alloc((size_t)words, st));
    CBX_HIP(hipMemsetAsync(buf.ptr, 0, sizeof(T) * nb * V, st));
    CBX_HIP(hipMemsetAsync(touched.ptr, 0, sizeof(uint32_t) * words, st));
    for (int64_t t0 = 0; t0 < n_terms; t0 += nb) {
        const int64_t n = std::min(nb, n_terms - t0);
        k_acc3_draw<T, I, K, IN_OV><<<grid_for(4 * n_lines, D3_NT), D3_NT, 0, st>>>(buf.ptr, touched.ptr, lines, n_lines,
                                                                               terms, t0, n, v, max_val, flags);
        k_acc3_fold<T, I, OUT_OV><<<grid_for(n * V, D3_NT), D3_NT, 0, st>>>(out, buf.ptr, touched.ptr, frames, t0, n, v);
        k_clear_words<<<grid_for((n * V + 31) / 32, D3_NT), D3_NT, 0, st>>>(touched.ptr, (n * V + 31) / 32);
        CBX_HIP(hipGetLastError());
    }
    return CBX_OK;
}

template <typename T, typename I, int IN_OV, int OUT_OV>
static int accumulate3_k(int kernel, T *out, const T *lines, int64_t n_lines, const I *terms, const I *frames,
                         int64_t n_terms, const Vol3 &v, T max_val, int *flags, hipStream_t st)
{
#define CBX_ACC3(KK)                                                                                          \
    accumulate3_batches<T, I, KK, IN_OV, OUT_OV>(out, lines, n_lines, terms, frames, n_terms, v, max_val, flags, st)
    switch (kernel) {
    case K_BIWEIGHT: return CBX_ACC3(K_BIWEIGHT);
    case K_GAUSSIAN: return CBX_ACC3(K_GAUSSIAN);
    case K_PARABOLIC: return CBX_ACC3(K_PARABOLIC);
    case K_RECTANGULAR: return CBX_ACC3(K_RECTANGULAR);
    default: return CBX_ACC3(K_TRIANGULAR);
    }
#undef CBX_ACC3
}

template <typename T, typename I>
static int accumulate_lines3(T *out, int64_t n_frames, int64_t D, int64_t H, int64_t W, const T *lines,
                             int64_t n_lines, const I *terms, const I *frames, int64_t n_terms, T max_val, int kernel,
                             int in_overlap, int out_overlap, void *stream)
{
    if (in_overlap < 0 || in_overlap > 1 || out_overlap < 0 || out_overlap > 1)
        return fail(CBX_EVALUE, "Invalid in_overlap and out_overlap keywords");
    int rc = check_vol(n_frames, D, H, W, n_lines, kernel, 0);
    if (rc) return rc;
    if (n_terms < 0) return fail(CBX_EVALUE, "negative size");
    if (n_lines > 0 && !terms) return fail(CBX_EVALUE, "terms must not be NULL");
    if (n_terms > 0 && !frames) return fail(CBX_EVALUE, "frames must not be NULL");
    hipStream_t st = (hipStream_t)stream;
    Workspace ws(st);
    const bool same = in_overlap == out_overlap;
    DevBuf<I> comp;
    const int64_t n_chk = std::max(n_lines, n_terms);
    if (n_chk > 0) {
        DevBuf<int> bad;
        CBX_HIP(bad.alloc(2, st));
        CBX_HIP(hipMemsetAsync(bad.ptr, 0, 2 * sizeof(int), st));
        if (same && n_lines > 0) CBX_HIP(comp.alloc(n_lines, st));
        k_term_frames3<I><<<grid_for(n_chk, D3_NT), D3_NT, 0, st>>>(terms, frames, n_lines, n_terms, n_frames,
                                                                   comp.ptr, bad.ptr);
        CBX_HIP(hipGetLastError());
        uint64_t hv[2] = {0, 0};
        const void *src[2] = {bad.ptr, bad.ptr + 1};
        const int bytes[2] = {4, 4};
        CBX_HIP(read_device_values(st, 2, src, bytes, hv));
        if (hv[1]) return fail(CBX_EINDEX, "frames is outside of (0, n_frames)");
        if (hv[0]) return fail(CBX_EINDEX, "a term index is outside of (0, len(frames))");
    }
    if (n_lines == 0 || n_frames * D * H * W == 0) return CBX_OK;
    if (same) {
        // max/max: the term buffer starts at zero, so with max_val < 0 every
        // drawn voxel holds 0 when its term ends
        const T mv = (in_overlap == 1 && max_val < T(0)) ? T(0) : max_val;
        return draw3_run<T, I>(out, Vol3{n_frames, D, H, W}, lines, n_lines, comp.ptr, mv, kernel, in_overlap, st);
    }
    const Vol3 v{n_frames, D, H, W};
    DevBuf<int> flags;
    CBX_HIP(flags.alloc(1, st));
    if ((rc = validate3<T, I>(lines, n_lines, nullptr, v, flags.ptr, st))) return rc;
    {
        KernelTimer timer("accumulate3", st);
        if (in_overlap == 0)
            rc = accumulate3_k<T, I, 0, 1>(kernel, out, lines, n_lines, terms, frames, n_terms, v, max_val, flags.ptr, st);
        else
            rc = accumulate3_k<T, I, 1, 0>(kernel, out, lines, n_lines, terms, frames, n_terms, v, max_val, flags.ptr, st);
    }
    if (rc) return rc;
    int hv = 0;
    if ((rc = read_flags(flags.ptr, st, &hv))) return rc;
    return flags3_status(hv);
}

} // namespace cbx

extern "C" {

int cbx_draw_lines3_f32(float *out, int64_t n_frames, int64_t depth, int64_t height, int64_t width,
                        const float *lines, int64_t n_lines, const int32_t *idxs, float max_val, int kernel,
                        int overlap, void *stream)
{
    return cbx::draw_lines3<float, int32_t>(out, n_frames, depth, height, width, lines, n_lines, idxs, max_val, kernel,
                                            overlap, stream);
}

int cbx_draw_lines3_f64(double *out, int64_t n_frames, int64_t depth, int64_t height, int64_t width,
                        const double *lines, int64_t n_lines, const int64_t *idxs, double max_val, int kernel,
                        int overlap, void *stream)
{
    return cbx::draw_lines3<double, int64_t>(out, n_frames, depth, height, width, lines, n_lines, idxs, max_val,
                                             kernel, overlap, stream);
}

int cbx_accumulate_lines3_f32(float *out, int64_t n_frames, int64_t depth, int64_t height, int64_t width,
                              const float *lines, int64_t n_lines, const int32_t *terms, const int32_t *frames,
                              int64_t n_terms, float max_val, int kernel, int in_overlap, int out_overlap, void *stream)
{
    return cbx::accumulate_lines3<float, int32_t>(out, n_frames, depth, height, width, lines, n_lines, terms, frames,
                                                  n_terms, max_val, kernel, in_overlap, out_overlap, stream);
}

int cbx_accumulate_lines3_f64(double *out, int64_t n_frames, int64_t depth, int64_t height, int64_t width,
                              const double *lines, int64_t n_lines, const int64_t *terms, const int64_t *frames,
                              int64_t n_terms, double max_val, int kernel, int in_overlap, int out_overlap,
                              void *stream)
{
    return cbx::accumulate_lines3<double, int64_t>(out, n_frames, depth, height, width, lines, n_lines, terms, frames,
                                                   n_terms, max_val, kernel, in_overlap, out_overlap, stream);
}

} // extern "C"
