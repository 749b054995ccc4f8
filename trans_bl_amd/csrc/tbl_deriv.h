// Line arithmetic of the compact derivatives (tbl_deriv_kernels.hip describes the
// scheme), shared by the derivative kernels and the right-hand side's
// (tbl_drv.hip).
#pragma once

#include "tbl_relax.h"

namespace tbl {

using C = cx<double>;

// affine map of a line's scalar state: x -> m x + c
struct Map {
    double m, c;
};
// x after y
__device__ __forceinline__ Map after(const Map &x, const Map &y)
{
    return {x.m * y.m, __builtin_fma(x.m, y.c, x.c)};
}
template <int CTRL>
__device__ __forceinline__ Map dpp_map(const Map &x)
{
    return {dpp<CTRL>(1.0, x.m), dpp0<CTRL>(x.c)};
}
__device__ __forceinline__ Map shfl_map(const Map &x, int src, int G)
{
    return {__shfl(x.m, src, G), __shfl(x.c, src, G)};
}
// inclusive scans of the lanes' maps in lane order / reverse lane order: DPP
// inside 16-lane rows, shuffles between rows
template <int G>
__device__ __forceinline__ Map scan_maps_up(Map x, int lane)
{
    x = after(x, dpp_map<0x111>(x));
    x = after(x, dpp_map<0x112>(x));
    x = after(x, dpp_map<0x114>(x));
    x = after(x, dpp_map<0x118>(x));
    if (G >= 32) {
        const Map q = shfl_map(x, (lane & 32) + 15, G);
        if (lane & 16) x = after(x, q);
    }
    if (G == 64) {
        const Map h = shfl_map(x, 31, G);
        if (lane & 32) x = after(x, h);
    }
    return x;
}
template <int G>
__device__ __forceinline__ Map scan_maps_down(Map x, int lane)
{
    x = after(x, dpp_map<0x101>(x));
    x = after(x, dpp_map<0x102>(x));
    x = after(x, dpp_map<0x104>(x));
    x = after(x, dpp_map<0x108>(x));
    if (G >= 32) {
        const Map q = shfl_map(x, (lane & 32) + 16, G);
        if (!(lane & 16)) x = after(x, q);
    }
    if (G == 64) {
        const Map h = shfl_map(x, 32, G);
        if (!(lane & 32)) x = after(x, h);
    }
    return x;
}

// x: table entry of row i of n: converged rows share one, the last two have
// their own, rows past n the zero entry
__device__ __forceinline__ int tri_row(int i, int n)
{
    return i < n - 2 ? min(i, kTriRows - 4) : min(kTriRows - 3 + i - (n - 2), kTriRows - 1);
}

// One tridiagonal line held R rows per lane; u: the right-hand sides over bet
// on entry, the solution on exit.  p(r), g(r): the factors of the lane's row
// r.  Rows past the line's end lie behind row n - 1, whose g is 0: they reach
// no row before them.
template <int R, typename F>
__device__ __forceinline__ Map line_forward(double (&u)[R], F p)
{
    Map m{1.0, 0.0};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        m.c = __builtin_fma(-p(r), m.c, u[r]);
        m.m *= -p(r);
        u[r] = m.c;
    }
    return m;
}
template <int R, typename F>
__device__ __forceinline__ void line_forward_in(double (&u)[R], F p, double in)
{
    double h = 1.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        h *= -p(r);
        u[r] = __builtin_fma(h, in, u[r]);
    }
}
template <int R, typename F>
__device__ __forceinline__ Map line_backward(double (&u)[R], F g)
{
    Map m{1.0, 0.0};
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
        m.c = __builtin_fma(-g(r), m.c, u[r]);
        m.m *= -g(r);
        u[r] = m.c;
    }
    return m;
}
template <int R, typename F>
__device__ __forceinline__ void line_backward_in(double (&u)[R], F g, double in)
{
    double h = 1.0;
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
        h *= -g(r);
        u[r] = __builtin_fma(h, in, u[r]);
    }
}

// The two closure right-hand sides at a lane's end of the line (the start for
// lanes of the first half, else the end): e the outermost point, s the next,
// NE and NE + 1 terms in the reference's order over the values F[0], F[1], ...
// from that end inwards; w: their weights, the scale last (8 each)
struct Closure {
    double e, s;
};
template <int NE>
__device__ __forceinline__ Closure closure(const double *w, const double (&F)[7])
{
    double e = w[0] * F[0], s = w[8] * F[0];
#pragma unroll
    for (int q = 1; q < NE; ++q) e = e + w[q] * F[q];
#pragma unroll
    for (int q = 1; q <= NE; ++q) s = s + w[8 + q] * F[q];
    return {e * w[7], s * w[15]};
}
// the lane's closure points of u: rows 0, 1 or n - 1, n - 2
template <int R>
__device__ __forceinline__ void put_closure(double (&u)[R], const Closure &b, int i0, int n)
{
    if (i0 == 0) {
        u[0] = b.e;
        u[1] = b.s;
    }
    const int re = (n - 1) % R, rs = (n - 2) % R;     // uniform
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r == rs) u[r] = i0 + r == n - 2 ? b.s : u[r];
        if (r == re) u[r] = i0 + r == n - 1 ? b.e : u[r];
    }
}
// F and the weights' side for a lane whose first row is i0
__device__ __forceinline__ int closure_points(const double *P, int i0, int n, double (&F)[7])
{
    const bool end = i0 >= n / 2;
#pragma unroll
    for (int q = 0; q < 7; ++q) F[q] = P[end ? n - 1 - q : q];
    return end ? 16 : 0;
}

// Global rows go through buffer resources over the line (x) or the mode (y):
// an access past the range reads zero or is dropped, so no access needs a
// branch.  A plane holds two values each side of its rows, zero where nothing
// was read, so the stencil windows need no clamp.
// (The whole offset is in the vector operand: the range check does not cover
// a scalar offset past the range.)
template <bool NT>
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, unsigned off, C v)
{
    u32x4 x;
    __builtin_memcpy(&x, &v, sizeof(x));
    __builtin_amdgcn_raw_buffer_store_b128(x, r, off, 0, NT ? 2 : 0);
}
// a workgroup's tables: `n` doubles, loads issued here, into LDS by the result
template <int NT, int M>
struct TableCopy {
    double v[M];
    int n;
    __device__ __forceinline__ TableCopy(const double *src, int count, int t) : n(count)
    {
#pragma unroll
        for (int q = 0; q < M; ++q) v[q] = src[min(t + NT * q, n - 1)];
    }
    __device__ __forceinline__ void store(double *dst, int t) const
    {
#pragma unroll
        for (int q = 0; q < M; ++q)
            if (t + NT * q < n) dst[t + NT * q] = v[q];
    }
};

// One direction of an x-line's solves, R points per lane, W wavefronts per part:
// a with the first derivative's factors (D1), b with the second's (D2), the two
// interleaved.  ta, tb: their tables; row: the points' entries; tot: the part's
// 8 W doubles for the wavefronts' maps.  Incoming state of a lane: its
// wavefront's (0, or through the maps of the wavefronts before it) sent
// through the lanes before it.
template <int R, int W, bool D1, bool D2>
__device__ __forceinline__ void x_solve_dir(bool up, double (&a)[R], double (&b)[R],
                                            const double *ta, const double *tb,
                                            const int (&row)[R], double *tot, int w, int lane)
{
    const int field = (up ? 1 : 2) * kTriRows;
    double pa[R], pb[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if constexpr (D1) pa[r] = ta[field + row[r]];
        if constexpr (D2) pb[r] = tb[field + row[r]];
    }
    auto fa = [&](int r) { return pa[r]; };
    auto fb = [&](int r) { return pb[r]; };
    Map ma{1.0, 0.0}, mb{1.0, 0.0};
    if constexpr (D1) ma = up ? line_forward<R>(a, fa) : line_backward<R>(a, fa);
    if constexpr (D2) mb = up ? line_forward<R>(b, fb) : line_backward<R>(b, fb);
    if constexpr (D1) ma = up ? scan_maps_up<64>(ma, lane) : scan_maps_down<64>(ma, lane);
    if constexpr (D2) mb = up ? scan_maps_up<64>(mb, lane) : scan_maps_down<64>(mb, lane);
    double sa = 0.0, sb = 0.0;
    if constexpr (W > 1) {
        double *tt = tot + (up ? 0 : 4 * W);
        if (lane == (up ? 63 : 0)) {
            tt[4 * w] = ma.m;
            tt[4 * w + 1] = ma.c;
            tt[4 * w + 2] = mb.m;
            tt[4 * w + 3] = mb.c;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < W - 1; ++q) {
            const int s = up ? q : W - 1 - q;
            if (up ? s < w : s > w) {
                if constexpr (D1) sa = __builtin_fma(tt[4 * s], sa, tt[4 * s + 1]);
                if constexpr (D2) sb = __builtin_fma(tt[4 * s + 2], sb, tt[4 * s + 3]);
            }
        }
    }
    const bool first = lane == (up ? 0 : 63);
    if constexpr (D1) {
        const Map e = up ? dpp_map<0x138>(ma) : dpp_map<0x130>(ma);
        const double in = first ? sa : __builtin_fma(e.m, sa, e.c);
        up ? line_forward_in<R>(a, fa, in) : line_backward_in<R>(a, fa, in);
    }
    if constexpr (D2) {
        const Map e = up ? dpp_map<0x138>(mb) : dpp_map<0x130>(mb);
        const double in = first ? sb : __builtin_fma(e.m, sb, e.c);
        up ? line_forward_in<R>(b, fb, in) : line_backward_in<R>(b, fb, in);
    }
}

// right-hand sides over the pivots of a lane's R points of an x-line in the
// plane P: interior points rhsx, rhsxx in the reference's sums, over 12 dx or
// 4 dx^2 and the pivot in one multiplication; w: the part's wavefront
template <int R, bool D1, bool D2>
__device__ __forceinline__ void x_rows(double (&a)[R], double (&b)[R], const double *P,
                                       const double *tab, const int (&row)[R], int i0, int w,
                                       int nx)
{
    const double *ta = tab, *tb = tab + 3 * kTriRows, *tc = tab + 6 * kTriRows;
    double x[R + 4];
#pragma unroll
    for (int q = 0; q < R + 4; ++q) x[q] = P[i0 + q - 2];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if constexpr (D1) a[r] = (x[r + 4] - x[r] + 28.0 * (x[r + 3] - x[r + 1])) * ta[row[r]];
        if constexpr (D2)
            b[r] = (3.0 * (x[r + 4] + x[r]) + 48.0 * (x[r + 3] + x[r + 1]) - 102.0 * x[r + 2]) *
                   tb[row[r]];
    }
    // the wavefronts that hold the line's first or last two points
    if (w == 0 || (w + 1) * 64 * R > nx - 2) {
        double F[7];
        const int side = closure_points(P, i0, nx, F);
        if constexpr (D1) put_closure<R>(a, closure<5>(tc + side, F), i0, nx);
        if constexpr (D2) put_closure<R>(b, closure<6>(tc + 32 + side, F), i0, nx);
    }
}

// right-hand sides over the pivots of a lane's R rows from j0 of a y-column in
// the plane P; M: rows of the tables; fv: wall row 0 of the first derivative
template <int R, bool D1, bool D2>
__device__ __forceinline__ void y_rows(double (&a)[R], double (&b)[R], const double *P,
                                       const DerivArgs &A, const double *tab, int M, int j0,
                                       int fv)
{
    const int ny = A.ny;
    const double *ta = tab + j0, *tb = ta + 3 * M, *tc = tab + 6 * M;
    double x[R + 4];
#pragma unroll
    for (int q = 0; q < R + 4; ++q) x[q] = P[j0 + q - 2];
    const double *c1 = A.cp_fd, *c2 = A.cp_sd;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if constexpr (D1)
            a[r] = (c1[3] * x[r] + c1[4] * x[r + 1] + c1[5] * x[r + 2] + c1[6] * x[r + 3]
                    + c1[7] * x[r + 4]) * ta[r];
        if constexpr (D2)
            b[r] = (c2[3] * x[r] + c2[4] * x[r + 1] + c2[5] * x[r + 2] + c2[6] * x[r + 3]
                    + c2[7] * x[r + 4]) * tb[r];
    }
    double F[7];
    const int side = closure_points(P, j0, ny, F);
    if constexpr (D1) {
        Closure c = closure<5>(tc + side, F);
        if (fv && side == 0) c.e = 0.0;
        put_closure<R>(a, c, j0, ny);
    }
    if constexpr (D2) put_closure<R>(b, closure<6>(tc + 32 + side, F), j0, ny);
}

// their solves, G lanes per column and part, a and b one after the other in
// each direction
template <int G, int R, bool D1, bool D2>
__device__ __forceinline__ void y_solve(double (&a)[R], double (&b)[R], const double *tab, int j0,
                                        int lane)
{
    constexpr int M = G * R;
    const double *ta = tab + j0, *tb = ta + 3 * M;
    auto pa = [&](int r) { return ta[M + r]; };
    auto pb = [&](int r) { return tb[M + r]; };
    auto ga = [&](int r) { return ta[2 * M + r]; };
    auto gb = [&](int r) { return tb[2 * M + r]; };
    if constexpr (D1) {
        const Map e = dpp_map<0x138>(scan_maps_up<G>(line_forward<R>(a, pa), lane));
        line_forward_in<R>(a, pa, lane == 0 ? 0.0 : e.c);
    }
    if constexpr (D2) {
        const Map e = dpp_map<0x138>(scan_maps_up<G>(line_forward<R>(b, pb), lane));
        line_forward_in<R>(b, pb, lane == 0 ? 0.0 : e.c);
    }
    if constexpr (D1) {
        const Map e = dpp_map<0x130>(scan_maps_down<G>(line_backward<R>(a, ga), lane));
        line_backward_in<R>(a, ga, lane == G - 1 ? 0.0 : e.c);
    }
    if constexpr (D2) {
        const Map e = dpp_map<0x130>(scan_maps_down<G>(line_backward<R>(b, gb), lane));
        line_backward_in<R>(b, gb, lane == G - 1 ? 0.0 : e.c);
    }
}

// x shapes (R, W): the fewest wavefronts per part with at most 9 points per
// lane, then the fewest points (17 points per lane took the registers of the
// wavefronts that hide the recurrences' latency)
#define TBL_X_SHAPES(X) \
    X(2, 1) X(3, 1) X(5, 1) X(7, 1) X(9, 1) X(5, 2) X(7, 2) X(9, 2) X(7, 3) X(9, 3) X(7, 4) X(9, 4)
// columns of a y workgroup's tile, and the stride of a column's plane in it
constexpr int kDerivYCols = 8;
template <int TX>
__host__ __device__ constexpr int y_stride(int rows) { return rows + 32 / TX; }
// y shapes (G, R): the first that holds the rows; R odd (an even lane stride
// puts the lanes of a column on few banks: 97 rows as 32 x 4 took 252 us for
// both derivatives of 1025x97x128, as 16 x 7 149)
#define TBL_Y_SHAPES(X) \
    X(16, 3) X(16, 5) X(16, 7) X(16, 9) X(32, 5) X(32, 7) X(32, 9) X(64, 5) X(64, 7) X(64, 9)

// workgroups, one per x-line: a dimension's threads are counted in 32 bits, so from
// 2^20 lines on in rows of that many
inline dim3 line_grid(size_t lines)
{
    const size_t row = lines < (size_t{1} << 20) ? lines : size_t{1} << 20;
    return dim3(static_cast<unsigned>(row), static_cast<unsigned>((lines + row - 1) / row));
}
__device__ __forceinline__ unsigned line_index() { return (blockIdx.y << 20) + blockIdx.x; }

// longest x-line accepted (ptsx), below the 64 * 9 * 4 points the shapes hold
constexpr int kDerivMaxNx = 2112;
inline bool x_shape(int nx, int *R, int *W)
{
    bool found = false;
    if (nx > kDerivMaxNx) return false;
#define X(RR, WW)                                                                   \
    if (64 * RR * WW >= nx && (!found || WW < *W || (WW == *W && RR < *R))) {       \
        found = true;                                                               \
        *R = RR;                                                                    \
        *W = WW;                                                                    \
    }
    TBL_X_SHAPES(X)
#undef X
    return found;
}

}  // namespace tbl
