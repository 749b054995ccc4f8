// Compact finite-difference derivatives (derivs_par.f:80-177) on gfx950.
//
// Arrays are in the caller's layout: complex (nx, ny, K), x fastest.  Each
// kernel reads its input once, coalesced, into LDS and produces one or both
// derivatives of a direction from it (3 passes over memory for the pair).
// The schemes are real, so a line's real and imaginary parts are two
// independent lines: LDS holds them as two planes and a lane works on one
// part -- half the registers per row, so twice the wavefronts per SIMD hide
// the recurrences' latency.
//  * x (derparx/derparxx, rhsx/rhsxx + tridparx at one rank,
//    derivs_par.f:80-113, 259-397, 775-858): a workgroup per x-line (j, k), W
//    wavefronts per part, R consecutive points per lane.
//  * y (dery/deryy/deryfv, rhsy/rhsyy/rhsyfv + tridy, derivs_par.f:116-177,
//    400-611, 947-975): a workgroup holds a tile of 8 or 4 columns x all ny rows
//    of one mode; G lanes per column and part, R rows per lane.
// Results go back through LDS and out as coalesced rows.
//
// Thomas solve: u_j = r_j / bet_j - p_j u_{j-1} and x_j = u_j - g_j x_{j+1},
// p_j = a_j / bet_j, g_j = c_j / bet_j (gam_{j+1} of tridy), the factors from
// the host.  Each direction is a local solve from a zero state, a scan of the
// lanes' affine maps and the homogeneous response of the incoming state.  The
// interior rows' weights are constants (also in y: the grid's ratio is), so
// the factors converge within 64 rows to the last bit or its neighbour: in x
// every row beyond reads one entry (kTriRows in all), in y, where a row has its
// own metric, each its own.  The tables sit in LDS.
// (Read from global memory, as 6 lane-segmented loads per row or 3 of the
// short tables, the address and data units were 85-98 % busy.)
//
// Both derivatives of 1025x193x64 (608 MB, 116 us at the rate of a copy): x
// 230 -> 115 us, y 212 -> 160; of 2049x257x32 (809 MB): x 1526 -> 157, y 275 ->
// 193.  x is bound by memory; y's rows of 128 bytes, mostly on two cache lines
// each, keep it above that (three workgroups a CU instead of two: no faster).
#include <cstdint>

#include "tbl_deriv.h"

namespace tbl {

// x-lines: o1 = d/dx (D1), o2 = d2/dx2 (D2) of f.  Workgroup: one line, W
// wavefronts per part; LDS: the two planes (LP values each; their reads at a
// lane stride of R, odd but for the shortest lines, are conflict-free), the
// wavefronts' maps, the tables.  Interior points: rhsx, rhsxx in the
// reference's sums, over 12 dx or 4 dx^2 and the pivot in one multiplication.
// The stores stream (nt): whole cache lines that the launch does not read
// again (1025x193x64, both derivatives: 130 -> 116 us).
// From 3 wavefronts per part the registers are held to 4 wavefronts a SIMD: two
// workgroups a CU (2049x257x32: 276 -> 198 us; below that it only spilled).
template <int R, int W, bool D1, bool D2>
__device__ __forceinline__ void deriv_x_line(const DerivArgs &A, unsigned block, const C *f, C *o1, C *o2)
{
    constexpr int NT = 128 * W, N = (R + 1) / 2, LP = 64 * R * W + 4;
    __shared__ double planes[2 * LP], maps[16 * W], tab[kXTab];
    const int t = threadIdx.x, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int part = wv / W, w = wv % W;
    const int nx = A.nx;
    const size_t line = static_cast<size_t>(block) * nx;
    {
        const __amdgpu_buffer_rsrc_t fr = buf_rsrc(f + line, static_cast<size_t>(nx) * sizeof(C));
        C v[N];
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = buf_load(fr, (t + NT * q) * sizeof(C), 0.0);
        const TableCopy<NT, (kXTab + NT - 1) / NT> tc(A.xtab, kXTab, t);
#pragma unroll
        for (int q = 0; q < N; ++q)
            if ((q + 1) * NT <= 64 * R * W || wv < W) {
                planes[2 + t + NT * q] = v[q].re;
                planes[LP + 2 + t + NT * q] = v[q].im;
            }
        if (t < 8) planes[t / 4 * LP + (t % 4 < 2 ? t % 4 : LP - 4 + t % 4)] = 0.0;
        tc.store(tab, t);
    }
    __syncthreads();
    double *P = planes + part * LP + 2, *tot = maps + part * 8 * W;
    const int i0 = (w * 64 + lane) * R;
    double a[R], b[R];
    int row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = tri_row(i0 + r, nx);
    x_rows<R, D1, D2>(a, b, P, tab, row, i0, w, nx);
    x_solve_dir<R, W, D1, D2>(true, a, b, tab, tab + 3 * kTriRows, row, tot, w, lane);
    x_solve_dir<R, W, D1, D2>(false, a, b, tab, tab + 3 * kTriRows, row, tot, w, lane);
    // out through the planes (a plane's readers are its own part's wavefronts:
    // past the maps' barriers, or this wavefront itself)
    auto out = [&](const double (&u)[R], C *o) {
#pragma unroll
        for (int r = 0; r < R; ++r) P[i0 + r] = u[r];
        __syncthreads();
        const __amdgpu_buffer_rsrc_t ro = buf_rsrc(o + line, static_cast<size_t>(nx) * sizeof(C));
#pragma unroll
        for (int q = 0; q < N; ++q)
            if ((q + 1) * NT <= 64 * R * W || wv < W)
                buf_store<true>(ro, (t + NT * q) * sizeof(C),
                                C{planes[2 + t + NT * q], planes[LP + 2 + t + NT * q]});
    };
    if constexpr (D1) out(a, o1);
    if constexpr (D1 && D2) __syncthreads();
    if constexpr (D2) out(b, o2);
}

template <int R, int W, bool D1, bool D2>
__global__ void __launch_bounds__(128 * W, W >= 3 ? 4 : 1)
    deriv_x_kernel(DerivArgs A, const C *__restrict__ f, C *__restrict__ o1, C *__restrict__ o2)
{
    const unsigned line = line_index();
    if (line < static_cast<unsigned>(A.ny) * A.K) deriv_x_line<R, W, D1, D2>(A, line, f, o1, o2);
}

// y-lines: o1 = d/dy (fv: with the wall row forced, deryfv), o2 = d2/dy2 of f.
// Workgroup: TX columns x all rows of one mode, both parts, in LDS (column
// stride LP, 32 / TX past a multiple of 32 values: the TX columns x 32 / TX rows of
// half a wavefront's tile accesses fall on different banks); G lanes per column
// and part.  Interior rows: rhsy, rhsyy in the reference's sums, times the metric
// of the spacing the generator normalised to (v_qdy(j-2), v_qdy2(j-2, 1);
// 1-based j) over the pivot; every row has its own table entry, at a constant
// offset from the lane's first.  The stores do not stream: a row's 128 bytes
// are rarely one cache line (with nt 8 of 9 sizes were up to 50 % slower).
// 8 columns, 4 with 64 lanes each: 1024 threads are a CU's only workgroup, and its
// load, solve and store phases overlap with nothing (us, one derivative and both:
// 569x545x8 27.2, 38.8 with 8 columns, 21.9, 31.6 with 4; 1025x321x64 220, 368 and
// 175, 281)
__host__ __device__ constexpr int y_cols(int G) { return G == 64 ? 4 : kDerivYCols; }
template <int G, int R, bool D1, bool D2>
__device__ __forceinline__ void deriv_y_tile(const DerivArgs &A, int block, const C *f, C *o1, int fv,
                                             C *o2)
{
    constexpr int TX = y_cols(G), NT = 2 * TX * G, N = (R + 1) / 2, M = G * R, LP = y_stride<TX>(M);
    constexpr int NTAB = 6 * M + 64;
    extern __shared__ double ylds[];
    double *planes = ylds, *tab = ylds + 2 * TX * LP;
    const int nx = A.nx, ny = A.ny, t = threadIdx.x;
    // workgroup n takes tile (n mod 8) * ceil(B/8) + n / 8 of the B tiles
    // (x fastest, then mode): the hardware deals workgroups to the 8 XCDs
    // round-robin, so neighbouring tiles -- whose rows share the cache line
    // at their boundary -- run on one XCD and share its L2
    const int tiles_x = (nx + TX - 1) / TX;
    const int B = tiles_x * A.K, per = (B + 7) / 8;
    const int m = block % 8 * per + block / 8;
    if (m >= B) return;
    const int x0 = (m % tiles_x) * TX, k = m / tiles_x;
    const size_t plane = static_cast<size_t>(nx) * ny, mb = plane * k;
    // thread: column x0 + t % 8, rows t / 8 + 2 G q
    const int tx = t % TX, tj = t / TX;
    const unsigned off = x0 + tx < nx ? static_cast<unsigned>((tj * nx + x0 + tx) * sizeof(C)) : kBufOff;
    const unsigned step = 2 * G * nx * static_cast<unsigned>(sizeof(C));
    double *re = planes + tx * LP + 2 + tj, *im = re + TX * LP;
    {
        const __amdgpu_buffer_rsrc_t fr = buf_rsrc(f + mb, plane * sizeof(C));
        C v[N];
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = buf_load(fr, off + step * q, 0.0);
        const TableCopy<NT, (NTAB + NT - 1) / NT> tc(A.ytab + (fv ? NTAB : 0), NTAB, t);
#pragma unroll
        for (int q = 0; q < N; ++q)
            if ((q + 1) * 2 * G <= M || tj + 2 * G * q < M) {
                re[2 * G * q] = v[q].re;
                im[2 * G * q] = v[q].im;
            }
        if (t < 8 * TX) planes[t / 4 * LP + (t % 4 < 2 ? t % 4 : M + t % 4)] = 0.0;
        tc.store(tab, t);
    }
    __syncthreads();
    const int lane = t % G, col = t / G;       // col: column, then part
    const int j0 = lane * R;
    double *P = planes + col * LP + 2;
    double a[R], b[R];
    y_rows<R, D1, D2>(a, b, P, A, tab, M, j0, fv);
    y_solve<G, R, D1, D2>(a, b, tab, j0, lane);
    // out through the tile (a column's group of lanes lies in one wavefront
    // and is its only reader until the barrier)
    auto out = [&](const double (&u)[R], C *o) {
#pragma unroll
        for (int r = 0; r < R; ++r) P[j0 + r] = u[r];
        __syncthreads();
        const __amdgpu_buffer_rsrc_t ro = buf_rsrc(o + mb, plane * sizeof(C));
#pragma unroll
        for (int q = 0; q < N; ++q)
            if ((q + 1) * 2 * G <= M || tj + 2 * G * q < M)
                buf_store<false>(ro, off + step * q, C{re[2 * G * q], im[2 * G * q]});
    };
    if constexpr (D1) out(a, o1);
    if constexpr (D1 && D2) __syncthreads();
    if constexpr (D2) out(b, o2);
}

template <int G, int R, bool D1, bool D2>
__global__ void __launch_bounds__(2 * y_cols(G) * G) deriv_y_kernel(DerivArgs A, const C *__restrict__ f,
                                                         C *__restrict__ o1, int fv,
                                                         C *__restrict__ o2)
{
    deriv_y_tile<G, R, D1, D2>(A, static_cast<int>(blockIdx.x), f, o1, fv, o2);
}

// all four derivatives of a small grid in one launch: the first ybs blocks (a
// multiple of 8) are y-tiles, the others x-lines of one wavefront per part (the
// blocks' other wavefronts leave before any barrier)
template <int RX, int RY>
__global__ void __launch_bounds__(256) deriv_both_kernel(DerivArgs A, int ybs, const C *__restrict__ f,
                                                         C *__restrict__ dx, C *__restrict__ dxx,
                                                         C *__restrict__ dy, C *__restrict__ dyy)
{
    const int block = static_cast<int>(blockIdx.x);
    if (block < ybs)
        deriv_y_tile<16, RY, true, true>(A, block, f, dy, 0, dyy);
    else if (threadIdx.x < 128)
        deriv_x_line<RX, 1, true, true>(A, block - ybs, f, dx, dxx);
}

// y-lines of more than 64 * 9 rows: one thread per column, the forward sweep
// stored in the output and re-read by the backward sweep (tridy's order).
// d/dy (rhsy 400-449), d2/dy2 (rhsyy 552-611), d/dy with wall row 0
// (rhsyfv 504-549); kind 2, 3, 4
__global__ void __launch_bounds__(64) deriv_y_line_kernel(DerivArgs A, int kind, const C *f, C *out)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    const int k = blockIdx.y;
    if (i >= A.nx) return;
    const int nx = A.nx, n = A.ny;
    const C *fl = f + static_cast<size_t>(k) * nx * n + i;
    C *ol = out + static_cast<size_t>(k) * nx * n + i;
    const int tk = kind - 2 + 2;   // thomas table index (kinds 2..4)
    const double *ta = A.thomas + static_cast<size_t>(tk) * kThomasFields * A.nmax;
    const double *tb = ta + A.nmax, *tg = tb + A.nmax;
    const double *qdy = A.qdy, *qdy2 = A.qdy2;
#define FY(J) fl[static_cast<size_t>((J) - 1) * nx]
    C prev = {0, 0};
    for (int J = 1; J <= n; ++J) {
        C r;
        if (kind == 2 || kind == 4) {
            const double *sp = A.sp_fd, *cp = A.cp_fd, *pp = A.pp_fd, *lp = A.lp_fd;
            if (J == 1) {
                if (kind == 2) {
                    const double *fe = A.fp_e;
                    r = qdy[0] * (fe[1] * FY(1) + fe[2] * FY(2) + fe[3] * FY(3) + fe[4] * FY(4)
                                  + fe[5] * FY(5));
                } else {
                    r = {0, 0};
                }
            } else if (J == 2) {
                r = qdy[0] * (sp[3] * FY(1) + sp[4] * FY(2) + sp[5] * FY(3) + sp[6] * FY(4)
                              + sp[7] * FY(5) + sp[8] * FY(6));
            } else if (J <= n - 2) {
                r = qdy[J - 3] * (cp[3] * FY(J - 2) + cp[4] * FY(J - 1) + cp[5] * FY(J)
                                  + cp[6] * FY(J + 1) + cp[7] * FY(J + 2));
            } else if (J == n - 1) {
                r = qdy[n - 6] * (pp[3] * FY(n) + pp[4] * FY(n - 1) + pp[5] * FY(n - 2)
                                  + pp[6] * FY(n - 3) + pp[7] * FY(n - 4) + pp[8] * FY(n - 5));
            } else {
                r = qdy[n - 5] * (lp[2] * FY(n) + lp[3] * FY(n - 1) + lp[4] * FY(n - 2)
                                  + lp[5] * FY(n - 3) + lp[6] * FY(n - 4));
            }
        } else {
            const double *fp = A.fp_sd, *sp = A.sp_sd, *cp = A.cp_sd, *pp = A.pp_sd, *lp = A.lp_sd;
            if (J == 1) {
                r = (fp[2] * FY(1) + fp[3] * FY(2) + fp[4] * FY(3) + fp[5] * FY(4) + fp[6] * FY(5)
                     + fp[7] * FY(6)) * qdy2[0];
            } else if (J == 2) {
                r = (sp[3] * FY(1) + sp[4] * FY(2) + sp[5] * FY(3) + sp[6] * FY(4) + sp[7] * FY(5)
                     + sp[8] * FY(6) + sp[9] * FY(7)) * qdy2[0];
            } else if (J <= n - 2) {
                r = (cp[3] * FY(J - 2) + cp[4] * FY(J - 1) + cp[5] * FY(J) + cp[6] * FY(J + 1)
                     + cp[7] * FY(J + 2)) * qdy2[J - 3];
            } else if (J == n - 1) {
                r = (pp[3] * FY(n) + pp[4] * FY(n - 1) + pp[5] * FY(n - 2) + pp[6] * FY(n - 3)
                     + pp[7] * FY(n - 4) + pp[8] * FY(n - 5) + pp[9] * FY(n - 6)) * qdy2[n - 7];
            } else {
                r = (lp[2] * FY(n) + lp[3] * FY(n - 1) + lp[4] * FY(n - 2) + lp[5] * FY(n - 3)
                     + lp[6] * FY(n - 4) + lp[7] * FY(n - 5)) * qdy2[n - 6];
            }
        }
        const C u = (J == 1) ? r / tb[0] : (r - ta[J - 1] * prev) / tb[J - 1];
        ol[static_cast<size_t>(J - 1) * nx] = u;
        prev = u;
    }
#undef FY
    C nxt = prev;
    for (int j = n - 2; j >= 0; --j) {
        C *p = ol + static_cast<size_t>(j) * nx;
        const C v = *p - tg[j + 1] * nxt;
        *p = v;
        nxt = v;
    }
}


static int deriv_x(const DerivArgs &A, const C *f, C *o1, C *o2, hipStream_t st)
{
    int R = 0, W = 0;
    if (!x_shape(A.nx, &R, &W)) return TBL_ERR_GRID;
    const dim3 grid = line_grid(static_cast<size_t>(A.ny) * A.K);
#define X(RR, WW)                                                                              \
    if (R == RR && W == WW) {                                                                  \
        const dim3 block(128 * WW);                                                            \
        if (o1 && o2)                                                                          \
            hipLaunchKernelGGL((deriv_x_kernel<RR, WW, true, true>), grid, block, 0, st, A,    \
                               f, o1, o2);                                                     \
        else if (o1)                                                                           \
            hipLaunchKernelGGL((deriv_x_kernel<RR, WW, true, false>), grid, block, 0, st, A,   \
                               f, o1, o2);                                                     \
        else                                                                                   \
            hipLaunchKernelGGL((deriv_x_kernel<RR, WW, false, true>), grid, block, 0, st, A,   \
                               f, o1, o2);                                                     \
        return TBL_OK;                                                                         \
    }
    TBL_X_SHAPES(X)
#undef X
    return TBL_ERR_GRID;
}

// rows the y shape of ny holds (0: the one-thread-per-column kernel)
int deriv_y_rows(int ny, int *G, int *R)
{
    *G = *R = 0;
#define X(GG, RR)             \
    if (!*R && GG * RR >= ny) { \
        *G = GG;              \
        *R = RR;              \
    }
    TBL_Y_SHAPES(X)
#undef X
    return *G * *R;
}

// bytes of LDS of a y workgroup: the tile's planes and the tables
static size_t y_lds(int G, int rows)
{
    const size_t tx = y_cols(G);
    return (2 * tx * (rows + 32 / tx) + 6 * rows + 64) * sizeof(double);
}

static int deriv_y(const DerivArgs &A, const C *f, C *o1, int fv, C *o2, hipStream_t st)
{
    int G, R;
    const int rows = deriv_y_rows(A.ny, &G, &R);
    if (!R) {
        const dim3 g2((A.nx + 63) / 64, A.K);
        if (o1) hipLaunchKernelGGL(deriv_y_line_kernel, g2, dim3(64), 0, st, A, fv ? 4 : 2, f, o1);
        if (o2) hipLaunchKernelGGL(deriv_y_line_kernel, g2, dim3(64), 0, st, A, 3, f, o2);
        return TBL_OK;
    }
    const int tiles = (A.nx + y_cols(G) - 1) / y_cols(G) * A.K;
    const dim3 grid(static_cast<unsigned>((tiles + 7) / 8 * 8));
    const size_t lds = y_lds(G, rows);
#define X(GG, RR)                                                                               \
    if (G == GG && R == RR) {                                                                   \
        const dim3 block(2 * y_cols(GG) * GG);                                                              \
        if (o1 && o2)                                                                           \
            hipLaunchKernelGGL((deriv_y_kernel<GG, RR, true, true>), grid, block, lds, st, A,   \
                               f, o1, fv, o2);                                                  \
        else if (o1)                                                                            \
            hipLaunchKernelGGL((deriv_y_kernel<GG, RR, true, false>), grid, block, lds, st, A,  \
                               f, o1, fv, o2);                                                  \
        else                                                                                    \
            hipLaunchKernelGGL((deriv_y_kernel<GG, RR, false, true>), grid, block, lds, st, A,  \
                               f, o1, fv, o2);                                                  \
        return TBL_OK;                                                                          \
    }
    TBL_Y_SHAPES(X)
#undef X
    return TBL_ERR_GRID;
}

int deriv(const DerivArgs &A, int kind, const double *f, double *out, hipStream_t st)
{
    const C *fi = reinterpret_cast<const C *>(f);
    C *fo = reinterpret_cast<C *>(out);
    switch (kind) {
    case 0: return deriv_x(A, fi, fo, nullptr, st);
    case 1: return deriv_x(A, fi, nullptr, fo, st);
    case 2: return deriv_y(A, fi, fo, 0, nullptr, st);
    case 3: return deriv_y(A, fi, nullptr, 0, fo, st);
    case 4: return deriv_y(A, fi, fo, 1, nullptr, st);
    default: return TBL_ERR_ARG;
    }
}

// Small grids take all four derivatives in one launch: a launch costs 3-5 us of
// latency whatever its size, and the two kinds of blocks share the chip's last
// wave.  Two launches -> one, us: 65x33x2 7.4 -> 4.4, 129x33x4 8.3 -> 4.6,
// 385x97x8 14.2 -> 10.7, 513x129x16 (3104 blocks) 29.4 -> 23.7, 513x129x32
// (6208) 46.1 -> 41.0, 513x129x64 (12416) 77.2 -> 76.3; from there on nothing or
// a loss (129x129x256, 37376: 103 -> 121), the larger kernel's registers and LDS
// cost occupancy.  Longer lines' x-blocks would leave half of a y-block's
// threads' registers idle: they keep their own launches.
constexpr int kBothBlocks = 8192;
static bool derivs_both(const DerivArgs &A, const C *f, C *dx, C *dxx, C *dy, C *dyy, hipStream_t st)
{
    int RX, W, G, RY;
    const int rows = deriv_y_rows(A.ny, &G, &RY);
    if (!x_shape(A.nx, &RX, &W) || W != 1 || G != 16) return false;
    const long tiles = (A.nx + kDerivYCols - 1) / kDerivYCols * static_cast<long>(A.K);
    const long ybs = (tiles + 7) / 8 * 8, blocks = ybs + static_cast<long>(A.ny) * A.K;
    if (blocks > kBothBlocks) return false;
    const size_t lds = y_lds(G, rows);
#define XY(RRX, RRY)                                                                              \
    if (RX == RRX && RY == RRY) {                                                                 \
        hipLaunchKernelGGL((deriv_both_kernel<RRX, RRY>), dim3(static_cast<unsigned>(blocks)),    \
                           dim3(256), lds, st, A, static_cast<int>(ybs), f, dx, dxx, dy, dyy);    \
        return true;                                                                              \
    }
#define X(RRX) XY(RRX, 3) XY(RRX, 5) XY(RRX, 7) XY(RRX, 9)
    X(2) X(3) X(5) X(7) X(9)
#undef X
#undef XY
    return false;
}

// Where an output lies over the input or over one of the other direction, the
// order counts (x, then y, which has read all of f it needs): two launches.
static bool directions_apart(const DerivArgs &A, const double *f, const double *const (&x)[2],
                             const double *const (&y)[2])
{
    const size_t n = static_cast<size_t>(A.nx) * A.ny * A.K * sizeof(C);
    auto apart = [n](const double *p, const double *q) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(p), b = reinterpret_cast<uintptr_t>(q);
        return a + n <= b || b + n <= a;
    };
    for (const double *p : {x[0], x[1]})
        if (!apart(p, f) || !apart(p, y[0]) || !apart(p, y[1])) return false;
    return apart(y[0], f) && apart(y[1], f);
}

int derivs4(const DerivArgs &A, const double *f, double *dx, double *dxx, double *dy, double *dyy,
            hipStream_t st)
{
    const C *fi = reinterpret_cast<const C *>(f);
    int rc = TBL_OK;
    if (dx && dxx && dy && dyy && directions_apart(A, f, {dx, dxx}, {dy, dyy}) &&
        derivs_both(A, fi, reinterpret_cast<C *>(dx), reinterpret_cast<C *>(dxx),
                    reinterpret_cast<C *>(dy), reinterpret_cast<C *>(dyy), st))
        return TBL_OK;
    if (dx || dxx)
        rc = deriv_x(A, fi, reinterpret_cast<C *>(dx), reinterpret_cast<C *>(dxx), st);
    if (rc == TBL_OK && (dy || dyy))
        rc = deriv_y(A, fi, reinterpret_cast<C *>(dy), 0, reinterpret_cast<C *>(dyy), st);
    return rc;
}

int deriv_kernel_attributes()
{
    hipError_t e = hipSuccess;
    auto allow = [&](const void *fn) {
        const hipError_t r =
            hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (r != hipSuccess) e = r;
    };
#define X(GG, RR)                                                                  \
    allow(reinterpret_cast<const void *>(&deriv_y_kernel<GG, RR, true, true>));    \
    allow(reinterpret_cast<const void *>(&deriv_y_kernel<GG, RR, true, false>));   \
    allow(reinterpret_cast<const void *>(&deriv_y_kernel<GG, RR, false, true>));
    TBL_Y_SHAPES(X)
#undef X
    return e == hipSuccess ? TBL_OK : TBL_ERR_HIP;
}

}  // namespace tbl
