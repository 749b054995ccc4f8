// Right-hand side of the vorticity equations and the RK4 update of the
// reference's Goertler case (my_form 1): lterms_gv / nlterms_gv
// (nlterms_par.f:89-182) with the z transforms of f_to_p / p_to_f
// (303-428), the combination of drv_gv (main_par.f:1339-1403), the four
// stage updates (main_par.f:270-341) and the gv_pert disturbance rows; and
// the flat-plate form (my_form 0): lterms_fi / nlterms_fi (nlterms_par.f:
// 6-86) and drv_fi's combination (main_par.f:1264-1336).
//
// User layout (complex (nx, ny, K), x fastest); base-flow arrays real
// (nx, ny).  All kernels but the nonlinear one are point-wise and
// HBM-bound.  The nonlinear terms transform every (x, y) point's K modes to
// kphys points in z, multiply there and transform back, all in LDS
// (nlterms_kernel) -- the transform pair of the reference's packed real FFT
// (mode 0 real, the odd-even mode in mode 0's imaginary part), to rounding.
#include "tbl_rhs.h"

namespace tbl {

namespace {

using cxd = cx<double>;

__device__ __forceinline__ cxd mul_i(double s, cxd a) { return {-s * a.im, s * a.re}; }

// lterms_gv (nlterms_par.f:100-108) at one point
__device__ __forceinline__ void lin_terms(double uxb, double uyb, double wzb, cxd ux, cxd uy,
                                          cxd wx, cxd wy, cxd wz, cxd &a, cxd &b, cxd &c,
                                          cxd &d)
{
    a = uyb * wx - wy * uxb;
    b = uxb * wz + ux * wzb;
    c = -uyb * wz - uy * wzb;
    d = (2.0 * uxb) * ux;
}

// lterms_fi's mode 1 (nlterms_par.f:19-24): the disturbance of b and c
// taken against the base flow's own products
__device__ __forceinline__ void lin_terms_fi1(double uxb, double uyb, double wzb, cxd ux, cxd uy,
                                              cxd wx, cxd wy, cxd wz, cxd &a, cxd &b, cxd &c)
{
    const cxd dwz = {wz.re - wzb, wz.im}, dux = {ux.re - uxb, ux.im}, duy = {uy.re - uyb, uy.im};
    a = uyb * wx - wy * uxb;
    b = uxb * dwz + wzb * dux;
    c = -uyb * dwz - wzb * duy;
}

__global__ void lterms_kernel(RhsArgs r)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y, k = blockIdx.z;
    if (i >= r.nx) return;
    const size_t e2 = static_cast<size_t>(j) * r.nx + i;
    const size_t e = static_cast<size_t>(k) * r.nx * r.ny + e2;
    if (r.fi) {
        // lterms_fi: modes >= 2 as lterms_gv without d (nlterms_par.f:28-34)
        cxd d;
        if (k == 0)
            lin_terms_fi1(r.b.uxb[e2], r.b.uyb[e2], r.b.wzb[e2], r.ux[e], r.uy[e], r.wx[e],
                          r.wy[e], r.wz[e], r.a[e], r.bb[e], r.c[e]);
        else
            lin_terms(r.b.uxb[e2], r.b.uyb[e2], r.b.wzb[e2], r.ux[e], r.uy[e], r.wx[e],
                      r.wy[e], r.wz[e], r.a[e], r.bb[e], r.c[e], d);
        return;
    }
    lin_terms(r.b.uxb[e2], r.b.uyb[e2], r.b.wzb[e2], r.ux[e], r.uy[e], r.wx[e], r.wy[e],
              r.wz[e], r.a[e], r.bb[e], r.c[e], r.d[e]);
}

// ---- nlterms_gv / nlterms_fi ------------------------------------------------------
// DFT of R values in registers, exponent -2 pi i k q / R
template <int R>
__device__ __forceinline__ void dft(cxd (&x)[R])
{
    if constexpr (R == 2) {
        const cxd a = x[0], b = x[1];
        x[0] = a + b;
        x[1] = a - b;
    } else if constexpr (R == 4) {
        const cxd a = x[0] + x[2], b = x[0] - x[2], c = x[1] + x[3], d = x[1] - x[3];
        x[0] = a + c;
        x[2] = a - c;
        x[1] = {b.re + d.im, b.im - d.re};
        x[3] = {b.re - d.im, b.im + d.re};
    } else {
        cxd e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
        dft<4>(e);
        dft<4>(o);
        const double h = 0.70710678118654752440;
        const cxd t[4] = {o[0], {h * (o[1].re + o[1].im), h * (o[1].im - o[1].re)},
                          {o[2].im, -o[2].re}, {h * (o[3].im - o[3].re), -h * (o[3].re + o[3].im)}};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            x[q] = e[q] + t[q];
            x[q + 4] = e[q] - t[q];
        }
    }
}
__device__ __forceinline__ cxd conj_of(cxd a) { return {a.re, -a.im}; }

// LDS slot of element n of one point's sequence: a skipped slot every 8 keeps
// the butterflies' strided reads on all banks
__host__ __device__ constexpr int nl_slot(int n) { return n + (n >> 3); }
// points of a workgroup and sequence stride (complex): N * points = 1024, so 256
// threads hold one pair of modes each
template <int N>
struct NlShape {
    static constexpr int M = N / 2, P = 1024 / N, SEQ = (nl_slot(M - 1) + 1) * P;
    static constexpr int FR = M >= 4 ? 4 : 2;           // radix of the innermost pass
};
// radix of the pass on sub-length L: 8 while that leaves 4s
constexpr int nl_radix(int L) { return L % 64 == 32 || L >= 128 ? 8 : L == 8 ? 2 : 4; }

// In-place passes of NS sequences: decimation in frequency from sub-length L
// down to FR (natural order in, digit-reversed out), and its transpose back
template <int N, int NS, int L, bool UP>
__device__ __forceinline__ void nl_pass(cxd *x, const cxd *tw)
{
    using S = NlShape<N>;
    constexpr int R = nl_radix(L), J = L / R, B = S::M / R * S::P;   // butterflies a sequence
    for (int e = threadIdx.x; e < NS * B; e += 256) {
        const int p = e % S::P, b = e / S::P % (S::M / R), f = e / B;
        const int j = b % J, base = b / J * L + j;
        cxd *s = x + f * S::SEQ + p;
        cxd v[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            v[q] = s[nl_slot(base + q * J) * S::P];
            if (UP && q) v[q] = cmul(v[q], tw[j * q * (N / L)]);
        }
        dft<R>(v);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (!UP && q) v[q] = cmul(v[q], tw[j * q * (N / L)]);
            s[nl_slot(base + q * J) * S::P] = v[q];
        }
    }
    __syncthreads();
}
template <int N, int NS, int L>
__device__ __forceinline__ void nl_down(cxd *x, const cxd *tw)
{
    if constexpr (L > NlShape<N>::FR) {
        nl_pass<N, NS, L, false>(x, tw);
        nl_down<N, NS, L / nl_radix(L)>(x, tw);
    }
}
template <int N, int NS, int L>
__device__ __forceinline__ void nl_up(cxd *x, const cxd *tw)
{
    if constexpr (L > NlShape<N>::FR) {
        nl_up<N, NS, L / nl_radix(L)>(x, tw);
        nl_pass<N, NS, L, true>(x, tw);
    }
}

// nlterms_gv (FI: nlterms_fi, the first three products, no base-flow terms).
// Each field is a real sequence of N values in z: its even and odd values are
// one complex sequence of M = N / 2 (no field is mixed with another, so a
// small one keeps its own rounding), transformed in place in LDS.  The
// inverse ends in digit-reversed order, where the products need no order;
// its innermost pass, the products and the first pass back are one step in
// registers.  A thread keeps the modes m and M - m of a point from the load to
// the base-flow terms.  As a direct DFT (O(K N) per point, 65 GFLOP at
// 1025x193x64 with N = 128) this kernel was bound by FP64 arithmetic: 3466 us;
// as FFTs by its LDS passes and memory (10 fields of 203 MB): 619 us.  From N = 512
// a workgroup's two points, or one, read 32 or 16 bytes of each cache line: 513x97x200
// with N = 512 688 us for 305 of bytes (direct 16100), 513x97x42 with 1024 1320 (7370).
template <int N, bool FI>
__global__ void __launch_bounds__(256) nlterms_kernel(RhsArgs r)
{
    using S = NlShape<N>;
    constexpr int M = S::M, P = S::P, NQ = FI ? 3 : 4, FR = S::FR;
    extern __shared__ double sm[];
    cxd *X = reinterpret_cast<cxd *>(sm), *tw = X + 6 * S::SEQ;
    const int K = r.K, t = threadIdx.x;
    const size_t plane = static_cast<size_t>(r.nx) * r.ny;
    // neighbouring groups of points share cache lines: in a row on one XCD
    const int groups = static_cast<int>((plane + P - 1) / P), per = (groups + 7) / 8;
    const int grp = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (grp >= groups) return;
    const size_t p0 = static_cast<size_t>(grp) * P;
    // this thread's point and modes (item 0: modes 0 and M / 2)
    const int p = t % P, m1 = t / P, m2 = m1 ? M - m1 : M / 2;
    const bool live = p0 + p < plane;
    const size_t at = live ? p0 + p : plane - 1;
    const cxd *in[6] = {r.ux, r.uy, r.uz, r.wx, r.wy, r.wz};
    cxd c1[6], c2[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        c1[f] = m1 < K ? in[f][m1 * plane + at] : cxd{0.0, 0.0};
        c2[f] = m2 < K ? in[f][m2 * plane + at] : cxd{0.0, 0.0};
    }
    for (int e = t; e < N; e += 256) tw[e] = {r.tw[e], -r.tw[N + e]};
    __syncthreads();
    // synthesis: v_n = Re c_0 + (Im c_0 / 2)(-1)^n + sum_m Re(c_m e^{-2 pi i m n / N});
    // with A_m = c_m / 2, A_{N-m} its conjugate, the even values' spectrum is A_m +
    // A_{m+M}, the odd ones' (A_m - A_{m+M}) e^{-2 pi i m / N}
    const cxd w1 = tw[m1], w2 = tw[m2];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        cxd z1, z2;
        if (m1) {
            const cxd a = 0.5 * c1[f], b = 0.5 * c2[f];
            const cxd o1 = cmul(a - conj_of(b), w1), o2 = cmul(b - conj_of(a), w2);
            z1 = a + conj_of(b) + cxd{-o1.im, o1.re};
            z2 = b + conj_of(a) + cxd{-o2.im, o2.re};
        } else {
            const double a = c1[f].re, h = 0.5 * c1[f].im;
            z1 = {a + h, a - h};
            // m = M / 2 pairs with itself: Re c + i (i Im c)(-i) = c's conjugate pair
            const cxd b = 0.5 * c2[f], o2 = cmul(b - conj_of(b), w2);
            z2 = b + conj_of(b) + cxd{-o2.im, o2.re};
        }
        X[f * S::SEQ + nl_slot(m1) * P + p] = z1;
        if (M > 1) X[f * S::SEQ + nl_slot(m2) * P + p] = z2;
    }
    __syncthreads();
    nl_down<N, 6, M>(X, tw);
    for (int e = t; e < M / FR * P; e += 256) {
        cxd *s = X + nl_slot(e / P * FR) * P + e % P;       // FR divides 8: no skip inside
        cxd v[6][FR];
#pragma unroll
        for (int f = 0; f < 6; ++f) {
#pragma unroll
            for (int q = 0; q < FR; ++q) v[f][q] = s[f * S::SEQ + q * P];
            dft<FR>(v[f]);
        }
        // ux uy uz wx wy wz -> a = uy wx - ux wy, b = ux wz - uz wx,
        // c = uz wy - uy wz, d = ux ux (nlterms_par.f:152-159), conjugated: the
        // analysis has the opposite sign in the exponent
        cxd y[4][FR];
#pragma unroll
        for (int q = 0; q < FR; ++q) {
            const cxd ux = v[0][q], uy = v[1][q], uz = v[2][q], wx = v[3][q], wy = v[4][q], wz = v[5][q];
            y[0][q] = {uy.re * wx.re - ux.re * wy.re, -(uy.im * wx.im - ux.im * wy.im)};
            y[1][q] = {ux.re * wz.re - uz.re * wx.re, -(ux.im * wz.im - uz.im * wx.im)};
            y[2][q] = {uz.re * wy.re - uy.re * wz.re, -(uz.im * wy.im - uy.im * wz.im)};
            y[3][q] = {ux.re * ux.re, -(ux.im * ux.im)};
        }
#pragma unroll
        for (int f = 0; f < NQ; ++f) {
            dft<FR>(y[f]);
#pragma unroll
            for (int q = 0; q < FR; ++q) s[f * S::SEQ + q * P] = y[f][q];
        }
    }
    __syncthreads();
    nl_up<N, NQ, M>(X, tw);
    if (!live) return;
    // analysis: c_0 = (1/N) sum v_n (real), c_m = (2/N) sum v_n e^{+2 pi i m n / N}
    // from the even and odd values' transforms; entries below 1e-14 flushed
    // (nlterms_par.f:418-423); then the base-flow terms (nlterms_par.f:167-177)
    cxd *out[4] = {r.a, r.bb, r.c, r.d};
    cxd n1[4], n2[4];
    const double sc = 2.0 / static_cast<double>(N);
    auto flush = [](cxd z) -> cxd {
        return {fabs(z.re) < 1e-14 ? 0.0 : z.re, fabs(z.im) < 1e-14 ? 0.0 : z.im};
    };
#pragma unroll
    for (int f = 0; f < NQ; ++f) {
        const cxd u = conj_of(X[f * S::SEQ + nl_slot(m1) * P + p]);
        const cxd v = M > 1 ? conj_of(X[f * S::SEQ + nl_slot(m2) * P + p]) : cxd{0.0, 0.0};
        if (m1) {
            const cxd e = 0.5 * (u + conj_of(v)), d = 0.5 * (u - conj_of(v));
            const cxd o = cmul(cxd{d.im, -d.re}, conj_of(w1));
            n1[f] = flush(sc * (e + o));
            n2[f] = flush(sc * conj_of(e - o));
        } else {
            n1[f] = flush(cxd{0.5 * sc * (u.re + u.im), 0.0});
            n2[f] = flush(sc * v);
        }
    }
    const size_t e2 = p0 + p;
    auto put = [&](int m, const cxd (&c)[6], const cxd (&nl)[4]) {
        if (m >= K) return;
        const size_t e = static_cast<size_t>(m) * plane + e2;
        if (FI) {
            out[0][e] = nl[0];
            out[1][e] = nl[1];
            out[2][e] = nl[2];
            return;
        }
        cxd la, lb, lc, ld;
        lin_terms(r.b.uxb[e2], r.b.uyb[e2], r.b.wzb[e2], c[0], c[1], c[3], c[4], c[5], la, lb, lc, ld);
        out[0][e] = la + nl[0];
        out[1][e] = lb + nl[1];
        out[2][e] = lc + nl[2];
        out[3][e] = ld + nl[3];
    };
    put(m1, c1, n1);
    if (M > 1) put(m2, c2, n2);
}

// the kphys values (LDS: six half-length sequences and the twiddles, 72 KB at 1024
// whatever the number of modes; 256 threads hold at most 1024 values)
#define TBL_NL_SIZES(X) X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)

// drv_gv's combination (main_par.f:1380-1397), rows 2..ny
__global__ void drv_combine_kernel(DrvArgs r)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y + 1, k = blockIdx.z;
    if (i >= r.nx) return;
    const size_t e2 = static_cast<size_t>(j) * r.nx + i;
    const size_t e = static_cast<size_t>(k) * r.nx * r.ny + e2;
    const double kb = -static_cast<double>(k) * r.beta;      // v_kb = i kb
    const double k2 = -static_cast<double>(k) * static_cast<double>(k) * r.beta * r.beta;
    const double rre = r.rre, fy = r.fac_y;
    if (r.fi) {
        // drv_fi's combination (main_par.f:1317-1331): no curvature terms
        r.dv[0][e] = -r.dady[e] + mul_i(kb, r.bb[e]) + rre * (r.xx[e] + fy * r.xy[e] + k2 * r.wx[e]);
        r.dv[1][e] = -mul_i(kb, r.c[e]) + r.dadx[e] + rre * (r.yx[e] + fy * r.yy[e] + k2 * r.wy[e]);
        r.dv[2][e] = -r.dbdx[e] + r.dcdy[e] + rre * (r.zx[e] + fy * r.zy[e] + k2 * r.wz[e]);
        return;
    }
    const double vg = r.b.varg[e2], dvg = r.b.dvargdx[e2];
    const cxd d = r.d[e];
    r.dv[0][e] = -r.dady[e] + mul_i(kb, r.bb[e]) - vg * mul_i(kb, d)
               + rre * (r.xx[e] + fy * r.xy[e] + k2 * r.wx[e]);
    r.dv[1][e] = -mul_i(kb, r.c[e]) + r.dadx[e] + rre * (r.yx[e] + fy * r.yy[e] + k2 * r.wy[e]);
    r.dv[2][e] = -r.dbdx[e] + r.dcdy[e] + vg * r.dddx[e] + dvg * d
               + rre * (r.zx[e] + fy * r.zy[e] + k2 * r.wz[e]);
}

// the RK4 stage updates (main_par.f:270-341) on rows 2..ny-1, columns i >= 3
__global__ void rk_update_kernel(RkArgs r)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int j = blockIdx.y + 1;
    const int k = blockIdx.z % r.K, q = blockIdx.z / r.K;
    if (i >= r.nx) return;
    const size_t e = (static_cast<size_t>(k) * r.ny + j) * r.nx + i;
    cxd *w = r.w[q], *w1 = r.w1[q], *dv1 = r.dv1[q];
    const cxd *dv2 = r.dv2[q];
    if (r.stage == 1) {
        const cxd v = w[e];
        w1[e] = v;
        w[e] = v + dv1[e] * r.h;
    } else if (r.stage == 4) {
        w[e] = w1[e] + r.h * (dv1[e] + dv2[e]);
    } else {
        const cxd d2 = dv2[e];
        w[e] = w1[e] + d2 * r.h;
        dv1[e] = dv1[e] + 2.0 * d2;
    }
}

// gv_pert's rows (main_par.f:1602-1607): uy(i,1,k), d2uydx2(i,k), k >= 2
__global__ void pert_kernel(cxd *uy, cxd *d2, const cxd *pu, const cxd *pd, int nx, int ny,
                            int i0, int n)
{
    const int i = i0 + blockIdx.x * blockDim.x + threadIdx.x;
    const int k = blockIdx.y + 1;
    if (i >= i0 + n) return;
    const size_t e = static_cast<size_t>(k) * nx + i;
    uy[static_cast<size_t>(k) * ny * nx + i] = pu[e];
    d2[e] = pd[e];
}

}  // namespace

bool nlterms_fits(int N)
{
#define X(NN) \
    if (N == NN) return true;
    TBL_NL_SIZES(X)
#undef X
    return false;
}

int terms(const RhsArgs &r, int kphys, hipStream_t st)
{
    if (kphys == 0) {
        dim3 grid((r.nx + 255) / 256, r.ny, r.K);
        hipLaunchKernelGGL(lterms_kernel, grid, dim3(256), 0, st, r);
    } else {
        const size_t plane = static_cast<size_t>(r.nx) * r.ny;
#define X(N)                                                                                  \
    if (kphys == N) {                                                                         \
        const size_t groups = (plane + NlShape<N>::P - 1) / NlShape<N>::P;                    \
        const dim3 grid(static_cast<unsigned>((groups + 7) / 8 * 8));                         \
        const size_t lds = sizeof(cxd) * (6 * NlShape<N>::SEQ + N);                           \
        if (r.fi)                                                                             \
            hipLaunchKernelGGL((nlterms_kernel<N, true>), grid, dim3(256), lds, st, r);       \
        else                                                                                  \
            hipLaunchKernelGGL((nlterms_kernel<N, false>), grid, dim3(256), lds, st, r);      \
        return TBL_OK;                                                                        \
    }
        TBL_NL_SIZES(X)
#undef X
        return TBL_ERR_ARG;
    }
    return TBL_OK;
}

int drv_combine(const DrvArgs &r, hipStream_t st)
{
    dim3 grid((r.nx + 255) / 256, r.ny - 1, r.K);
    hipLaunchKernelGGL(drv_combine_kernel, grid, dim3(256), 0, st, r);
    return TBL_OK;
}

int rk_update(const RkArgs &r, hipStream_t st)
{
    if (r.nx <= 2 || r.ny <= 2) return TBL_OK;
    dim3 grid((r.nx - 2 + 255) / 256, r.ny - 2, 3 * r.K);
    hipLaunchKernelGGL(rk_update_kernel, grid, dim3(256), 0, st, r);
    return TBL_OK;
}

int pert_rows(cx<double> *uy, cx<double> *d2, const cx<double> *pu, const cx<double> *pd,
              int nx, int ny, int K, int i0, int i1, hipStream_t st)
{
    const int n = i1 - i0 + 1;
    if (n <= 0 || K < 2) return TBL_OK;
    dim3 grid((n + 63) / 64, K - 1);
    hipLaunchKernelGGL(pert_kernel, grid, dim3(64), 0, st, uy, d2, pu, pd, nx, ny, i0, n);
    return TBL_OK;
}

int rhs_kernel_attributes()
{
#define X(N)                                                                                       \
    TBL_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&nlterms_kernel<N, false>),         \
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));          \
    TBL_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&nlterms_kernel<N, true>),          \
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    TBL_NL_SIZES(X)
#undef X
    return TBL_OK;
}

}  // namespace tbl
