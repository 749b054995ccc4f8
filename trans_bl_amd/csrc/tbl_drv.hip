// The right-hand side's combination of terms and derivatives (drv_gv,
// main_par.f:1339-1403; drv_fi, main_par.f:1264-1336) on gfx950, derivative
// solves included: per component one launch over the y-lines, which leaves the
// y-derivatives' share in dv, and one over the x-lines, which adds the
// x-derivatives and the pointwise terms:
//   dvx = [-da/dy + (fac_y/Re) d2wx/dy2] + d2wx/dx2 / Re + k2 wx / Re + i kb (b - vg d)
//   dvy = [(fac_y/Re) d2wy/dy2]          + d2wy/dx2 / Re + k2 wy / Re - i kb c + da/dx
//   dvz = [dc/dy + (fac_y/Re) d2wz/dy2]  + d2wz/dx2 / Re + k2 wz / Re - db/dx + vg dd/dx + dvg d
// No derivative is stored, and the linear terms (LIN: lterms_gv,
// nlterms_par.f:100-108) are formed where they are used from the fields and the
// base flow, whose (nx, ny) arrays stay in the caches over the modes.
//
// Bound by memory: 23 passes over a field of the (nx, ny, K) grid, linear terms
// included, against 51 with the terms, the eleven derivatives and their
// combination in kernels of their own (42 with stored nonlinear terms).
// 1025x193x64, of the terms' output on: 1606 us in the separate kernels, 1015
// here (x 176-231 us per component at 4.4-5.7 TB/s, y 161 at 3.8 and 85); with
// linear terms 1960 -> 1010.
// The line arithmetic and the layout in LDS are the derivative kernels'
// (tbl_deriv_kernels.hip); a line's second input follows the first through the
// same planes, so the workgroups per CU stay; the registers are held to 4
// wavefronts a SIMD from 2 wavefronts per part (140 -> 128; below that it spilled).
#include "tbl_deriv.h"
#include "tbl_rhs.h"

namespace tbl {

namespace {

__device__ __forceinline__ C times_i(double s, C a) { return {-s * a.im, s * a.re}; }

// y share of component Q, dv = s1 df1/dy + s2 d2w/dy2, all rows but the first:
// f1 = a (Q 0), c (Q 2), stored or LIN; Q 1 has no f1
template <int G, int R, int Q, bool LIN>
__global__ void __launch_bounds__(16 * G) drv_y_kernel(DerivArgs A, DrvArgs r)
{
    constexpr int TX = kDerivYCols, NT = 2 * TX * G, N = (R + 1) / 2, M = G * R, LP = M + 4;
    constexpr int NTAB = 6 * M + 64;
    constexpr bool F1 = Q != 1;
    extern __shared__ double ylds[];
    double *planes = ylds, *tab = ylds + 2 * TX * LP;
    const int nx = A.nx, t = threadIdx.x;
    // neighbouring tiles on one XCD, as in deriv_y_kernel
    const int tiles_x = (nx + TX - 1) / TX;
    const int B = tiles_x * A.K, per = (B + 7) / 8;
    const int m = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (m >= B) return;
    const int x0 = (m % tiles_x) * TX, k = m / tiles_x;
    const size_t plane = static_cast<size_t>(nx) * A.ny, mb = plane * k;
    const int tx = t % TX, tj = t / TX;
    const unsigned off = x0 + tx < nx ? static_cast<unsigned>((tj * nx + x0 + tx) * sizeof(C)) : kBufOff;
    const unsigned step = 2 * G * nx * static_cast<unsigned>(sizeof(C));
    double *re = planes + tx * LP + 2 + tj, *im = re + TX * LP;
    auto put = [&](const C (&v)[N]) {
#pragma unroll
        for (int q = 0; q < N; ++q)
            if ((q + 1) * 2 * G <= M || tj + 2 * G * q < M) {
                re[2 * G * q] = v[q].re;
                im[2 * G * q] = v[q].im;
            }
    };
    const int lane = t % G, col = t / G, j0 = lane * R;
    double *P = planes + col * LP + 2;
    double a[R], b[R];
    {
        auto load = [&](const C *p, C (&v)[N]) {
            const __amdgpu_buffer_rsrc_t s = buf_rsrc(p + mb, plane * sizeof(C));
#pragma unroll
            for (int q = 0; q < N; ++q) v[q] = buf_load(s, off + step * q, 0.0);
        };
        C v1[N], v2[N];
        load(Q == 0 ? r.wx : Q == 1 ? r.wy : r.wz, v2);
        if constexpr (F1 && !LIN) load(Q == 0 ? r.a : r.c, v1);
        if constexpr (F1 && LIN) {
            // a = uyb wx - wy uxb; c = -(uyb wz + uy wzb)
            load(Q == 0 ? r.wy : r.uy, v1);
            const __amdgpu_buffer_rsrc_t sp = buf_rsrc(r.b.uyb, plane * sizeof(double));
            const __amdgpu_buffer_rsrc_t sq = buf_rsrc(Q == 0 ? r.b.uxb : r.b.wzb, plane * sizeof(double));
            double bp[N], bq[N];
#pragma unroll
            for (int q = 0; q < N; ++q) {
                bp[q] = buf_scalar(sp, (off + step * q) / 2, 0.0);
                bq[q] = buf_scalar(sq, (off + step * q) / 2, 0.0);
            }
#pragma unroll
            for (int q = 0; q < N; ++q)
                v1[q] = Q == 0 ? bp[q] * v2[q] - v1[q] * bq[q] : bp[q] * v2[q] + v1[q] * bq[q];
        }
        const TableCopy<NT, (NTAB + NT - 1) / NT> tc(A.ytab, NTAB, t);
        put(F1 ? v1 : v2);
        if (t < 64) planes[t / 4 * LP + (t % 4 < 2 ? t % 4 : M + t % 4)] = 0.0;
        tc.store(tab, t);
        __syncthreads();
        if constexpr (F1) {
            y_rows<R, true, false>(a, b, P, A, tab, M, j0, 0);
            __syncthreads();
            put(v2);
            __syncthreads();
        }
    }
    y_rows<R, false, true>(a, b, P, A, tab, M, j0, 0);
    y_solve<G, R, F1, true>(a, b, tab, j0, lane);
    const double s1 = Q == 0 || LIN ? -1.0 : 1.0, s2 = r.rre * r.fac_y;
#pragma unroll
    for (int q = 0; q < R; ++q) P[j0 + q] = F1 ? s1 * a[q] + s2 * b[q] : s2 * b[q];
    __syncthreads();
    const __amdgpu_buffer_rsrc_t ro = buf_rsrc(r.dv[Q] + mb, plane * sizeof(C));
#pragma unroll
    for (int q = 0; q < N; ++q)
        if ((q + 1) * 2 * G <= M || tj + 2 * G * q < M)
            buf_store<false>(ro, tj + q == 0 ? kBufOff : off + step * q, C{re[2 * G * q], im[2 * G * q]});
}

// x share of component Q and the pointwise terms onto dv; lines of rows 1..
template <int R, int W, int Q, bool LIN>
__global__ void __launch_bounds__(128 * W, W >= 2 ? 4 : 1) drv_x_kernel(DerivArgs A, DrvArgs r)
{
    constexpr int NT = 128 * W, N = (R + 1) / 2, LP = 64 * R * W + 4;
    constexpr bool F1 = Q != 0;
    __shared__ double planes[2 * LP], maps[16 * W], tab[kXTab];
    const int t = threadIdx.x, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int part = wv / W, w = wv % W;
    const int nx = A.nx, rows = A.ny - 1, m = static_cast<int>(line_index()), k = m / rows, j = 1 + m % rows;
    if (k >= A.K) return;
    const size_t line = (static_cast<size_t>(k) * A.ny + j) * nx, line2 = static_cast<size_t>(j) * nx;
    auto load = [&](const C *p, C (&v)[N]) {
        const __amdgpu_buffer_rsrc_t s = buf_rsrc(p + line, static_cast<size_t>(nx) * sizeof(C));
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = buf_load(s, (t + NT * q) * sizeof(C), 0.0);
    };
    auto load2 = [&](const double *p, double (&v)[N]) {
        const __amdgpu_buffer_rsrc_t s = buf_rsrc(p + line2, static_cast<size_t>(nx) * sizeof(double));
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = buf_scalar(s, (t + NT * q) * sizeof(double), 0.0);
    };
    auto put = [&](const C (&v)[N]) {
#pragma unroll
        for (int q = 0; q < N; ++q)
            if ((q + 1) * NT <= 64 * R * W || wv < W) {
                planes[2 + t + NT * q] = v[q].re;
                planes[LP + 2 + t + NT * q] = v[q].im;
            }
    };
    double *P = planes + part * LP + 2, *tot = maps + part * 8 * W;
    const double *ta = tab, *tb = tab + 3 * kTriRows;
    const int i0 = (w * 64 + lane) * R;
    const double rre = r.rre, kb = -static_cast<double>(k) * r.beta;      // v_kb = i kb
    const double k2 = -static_cast<double>(k) * static_cast<double>(k) * r.beta * r.beta;
    double a[R], b[R];
    int row[R];
#pragma unroll
    for (int q = 0; q < R; ++q) row[q] = tri_row(i0 + q, nx);
    {
        // v1: the first derivative's input (a, b), v2: the vorticity
        C v1[N], v2[N];
        load(Q == 0 ? r.wx : Q == 1 ? r.wy : r.wz, v2);
        if constexpr (F1 && !LIN) load(Q == 1 ? r.a : r.bb, v1);
        if constexpr (F1 && LIN) {
            double f[N], g[N];
            load(Q == 1 ? r.wx : r.ux, v1);
            load2(Q == 1 ? r.b.uyb : r.b.uxb, f);
            load2(Q == 1 ? r.b.uxb : r.b.wzb, g);
#pragma unroll
            for (int q = 0; q < N; ++q)
                v1[q] = Q == 1 ? f[q] * v1[q] - v2[q] * g[q] : f[q] * v2[q] + v1[q] * g[q];
        }
        const TableCopy<NT, (kXTab + NT - 1) / NT> tc(A.xtab, kXTab, t);
        put(F1 ? v1 : v2);
        if (t < 8) planes[t / 4 * LP + (t % 4 < 2 ? t % 4 : LP - 4 + t % 4)] = 0.0;
        tc.store(tab, t);
        __syncthreads();
        if constexpr (F1) {
            x_rows<R, true, false>(a, b, P, tab, row, i0, w, nx);
            __syncthreads();
            put(v2);
            __syncthreads();
        }
    }
    x_rows<R, false, true>(a, b, P, tab, row, i0, w, nx);
    x_solve_dir<R, W, F1, true>(true, a, b, ta, tb, row, tot, w, lane);
    x_solve_dir<R, W, F1, true>(false, a, b, ta, tb, row, tot, w, lane);
    // the x share, k2 w from the plane included, to point order (a plane's
    // readers as in deriv_x_kernel); what dv holds; the pointwise terms
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const double v = rre * (b[q] + k2 * P[i0 + q]);
        P[i0 + q] = Q == 0 ? v : Q == 1 ? a[q] + v : v - a[q];
    }
    C s[N], v3[N];
    load(r.dv[Q], s);
    if constexpr (Q == 0) {
        // i kb (b - vg d)
        C e[N];
        if constexpr (LIN) {
            double p[N], q2[N], vg[N];
            load(r.wz, e);
            load(r.ux, v3);
            load2(r.b.uxb, p);
            load2(r.b.wzb, q2);
            load2(r.b.varg, vg);
#pragma unroll
            for (int q = 0; q < N; ++q)
                e[q] = (p[q] * e[q] + v3[q] * q2[q]) - vg[q] * ((2.0 * p[q]) * v3[q]);
        } else {
            load(r.bb, e);
            if (!r.fi) {
                double vg[N];
                load(r.d, v3);
                load2(r.b.varg, vg);
#pragma unroll
                for (int q = 0; q < N; ++q) e[q] = e[q] - vg[q] * v3[q];
            }
        }
#pragma unroll
        for (int q = 0; q < N; ++q) s[q] = s[q] + times_i(kb, e[q]);
    }
    if constexpr (Q == 1) {
        C e[N];
        if constexpr (LIN) {
            double p[N], q2[N];
            load(r.wz, e);
            load(r.uy, v3);
            load2(r.b.uyb, p);
            load2(r.b.wzb, q2);
#pragma unroll
            for (int q = 0; q < N; ++q) e[q] = p[q] * e[q] + v3[q] * q2[q];      // -c
        } else {
            load(r.c, e);
        }
#pragma unroll
        for (int q = 0; q < N; ++q) s[q] = s[q] + times_i(LIN ? kb : -kb, e[q]);
    }
    auto get = [&](int q) -> C {
        if ((q + 1) * NT <= 64 * R * W || wv < W)
            return {planes[2 + t + NT * q], planes[LP + 2 + t + NT * q]};
        return {0.0, 0.0};
    };
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; ++q) s[q] = s[q] + get(q);
    if (Q == 2 && !r.fi) {
        double vg[N], dvg[N];
        load(LIN ? r.ux : r.d, v3);
        if constexpr (LIN) {
            load2(r.b.uxb, vg);
#pragma unroll
            for (int q = 0; q < N; ++q) v3[q] = (2.0 * vg[q]) * v3[q];
        }
        load2(r.b.varg, vg);
        load2(r.b.dvargdx, dvg);
        __syncthreads();
        put(v3);
        __syncthreads();
        x_rows<R, true, false>(a, b, P, tab, row, i0, w, nx);
        x_solve_dir<R, W, true, false>(true, a, b, ta, tb, row, tot, w, lane);
        x_solve_dir<R, W, true, false>(false, a, b, ta, tb, row, tot, w, lane);
#pragma unroll
        for (int q = 0; q < R; ++q) P[i0 + q] = a[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < N; ++q) s[q] = s[q] + vg[q] * get(q) + dvg[q] * v3[q];
    }
    const __amdgpu_buffer_rsrc_t ro = buf_rsrc(r.dv[Q] + line, static_cast<size_t>(nx) * sizeof(C));
#pragma unroll
    for (int q = 0; q < N; ++q)
        if ((q + 1) * NT <= 64 * R * W || wv < W) buf_store<true>(ro, (t + NT * q) * sizeof(C), s[q]);
}

template <int Q, bool LIN>
void launch_y(const DerivArgs &A, const DrvArgs &r, hipStream_t st)
{
    int G, R;
    const int rows = deriv_y_rows(A.ny, &G, &R);
    const int tiles = (A.nx + kDerivYCols - 1) / kDerivYCols * A.K;
    const dim3 grid(static_cast<unsigned>((tiles + 7) / 8 * 8));
    const size_t lds =
        (static_cast<size_t>(2 * kDerivYCols) * (rows + 4) + 6 * rows + 64) * sizeof(double);
#define X(GG, RR)           \
    if (G == GG && R == RR) \
        hipLaunchKernelGGL((drv_y_kernel<GG, RR, Q, LIN>), grid, dim3(16 * GG), lds, st, A, r);
    TBL_Y_SHAPES(X)
#undef X
}

template <int Q, bool LIN>
void launch_x(const DerivArgs &A, const DrvArgs &r, hipStream_t st)
{
    int R = 0, W = 0;
    x_shape(A.nx, &R, &W);
    const dim3 grid = line_grid(static_cast<size_t>(A.ny - 1) * A.K);
#define X(RR, WW)           \
    if (R == RR && W == WW) \
        hipLaunchKernelGGL((drv_x_kernel<RR, WW, Q, LIN>), grid, dim3(128 * WW), 0, st, A, r);
    TBL_X_SHAPES(X)
#undef X
}

template <bool LIN>
void launch_all(const DerivArgs &A, const DrvArgs &r, hipStream_t st)
{
    launch_y<0, LIN>(A, r, st);
    launch_x<0, LIN>(A, r, st);
    launch_y<1, LIN>(A, r, st);
    launch_x<1, LIN>(A, r, st);
    launch_y<2, LIN>(A, r, st);
    launch_x<2, LIN>(A, r, st);
}

}  // namespace

bool drv_fused_fits(const DerivArgs &A)
{
    int a, b;
    return x_shape(A.nx, &a, &b) && deriv_y_rows(A.ny, &a, &b) && A.ny > 1;
}

int drv_fused(const DerivArgs &A, const DrvArgs &r, bool lin, hipStream_t st)
{
    if (!drv_fused_fits(A) || (lin && r.fi)) return TBL_ERR_ARG;
    if (lin)
        launch_all<true>(A, r, st);
    else
        launch_all<false>(A, r, st);
    return TBL_OK;
}

int drv_kernel_attributes()
{
    hipError_t e = hipSuccess;
    auto allow = [&](const void *fn) {
        const hipError_t q =
            hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (q != hipSuccess) e = q;
    };
#define Y(GG, RR, Q)                                                         \
    allow(reinterpret_cast<const void *>(&drv_y_kernel<GG, RR, Q, true>));   \
    allow(reinterpret_cast<const void *>(&drv_y_kernel<GG, RR, Q, false>));
#define X(GG, RR) Y(GG, RR, 0) Y(GG, RR, 1) Y(GG, RR, 2)
    TBL_Y_SHAPES(X)
#undef X
#undef Y
    return e == hipSuccess ? TBL_OK : TBL_ERR_HIP;
}

}  // namespace tbl
