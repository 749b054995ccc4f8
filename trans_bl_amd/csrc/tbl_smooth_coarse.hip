// Coarsest-level smoother: every sweep of the level in one launch, one
// workgroup per mode with the level resident in LDS.
#include <algorithm>
#include <type_traits>

#include "tbl_relax.h"

namespace tbl {

// Coarsest level: one workgroup per mode keeps the whole level in LDS and
// runs every sweep (20*itera, poisson_par.f:45) without leaving the CU.  LDS
// holds v with a compact odd column stride and the mode's line-LU factors;
// the source is read from global memory.  (Scan form, for levels whose lines
// are too long for the one-thread-per-line kernel below.)
__host__ __device__ inline int coarse_stride(int ny) { return ny | 1; }

template <typename T>
__host__ __device__ inline size_t coarse_lds_bytes(int nx, int ny, bool with_s)
{
    const size_t col = static_cast<size_t>(coarse_stride(ny)) * nx * sizeof(cx<T>);
    return col * (with_s ? 2 : 1) + static_cast<size_t>(2 * kLuFields) * ny * sizeof(T);
}

template <typename T, int G, int R>
__global__ void __launch_bounds__(512) smooth_coarsest_kernel(LevelArgs<T> L, cx<T> *V,
                                                               const cx<T> *S, const T *lu,
                                                               int sweeps, T rf,
                                                               const int *active)
{
    extern __shared__ unsigned char smem_raw[];
    const int k = blockIdx.x;
    if (active && !active[k]) return;
    const int nx = L.nx, ny = L.ny, ld = L.ld, ls = coarse_stride(ny);
    cx<T> *sv = reinterpret_cast<cx<T> *>(smem_raw);
    T *slu = reinterpret_cast<T *>(sv + static_cast<size_t>(ls) * nx);
    cx<T> *gv = V + static_cast<size_t>(k) * L.plane;
    const cx<T> *gs = S + static_cast<size_t>(k) * L.plane;
    const T *glu = lu + (static_cast<size_t>(k) * 2) * kLuFields * L.lus;
    for (int e = threadIdx.x; e < nx * ny; e += blockDim.x) {
        const int i = e / ny, j = e % ny;
        sv[i * ls + j] = gv[static_cast<size_t>(i) * ld + j];
    }
    for (int e = threadIdx.x; e < 2 * kLuFields * ny; e += blockDim.x)
        slu[e] = glu[static_cast<size_t>(e / ny) * L.lus + e % ny];
    __syncthreads();
    // the line solve indexes the factors with stride L.ld: give it ny here
    LevelArgs<T> Ls = L;
    Ls.ld = ny;
    const int groups = blockDim.x / G;
    const int grp = threadIdx.x / G, lane = threadIdx.x % G;
    for (int it = 0; it < sweeps; ++it) {
        for (int phase = 0; phase < 4; ++phase) {
            const int nl = phase_lines(phase, nx);
            for (int c = grp; c < nl; c += groups) {
                const int i = phase_column(phase, c, nx);
                const int side = (phase == 0) ? (c == 0 ? -1 : 1) : 0;
                cx<T> *col = sv + static_cast<size_t>(i) * ls;
                const cx<T> *scol = gs + static_cast<size_t>(i) * ld;
                const LineLU<T, R> f =
                    load_line_lu<T, R>(slu + (side ? kLuFields * ny : 0), ny, line_j0(lane, R), ny);
                relax_core<T, G, R>(
                    Ls, f, rf, lane,
                    [&](int j) { return xoff<T>(col, ls, j, side, side == 0 && j >= ny - 2); },
                    [&](int j) { return col[j]; }, [&](int j, int) { return scol[j]; },
                    [&](int j, cx<T> v) { col[j] = v; });
            }
            __syncthreads();
        }
    }
    for (int e = threadIdx.x; e < nx * ny; e += blockDim.x) {
        const int i = e / ny, j = e % ny;
        gv[static_cast<size_t>(i) * ld + j] = sv[i * ls + j];
    }
}

// Coarsest level through the inverses of its line matrices.  A line's matrix
// depends only on the mode and on centre/border (coef_center / coef_border,
// poisson_par.f:229-340), so one relaxation of every line of a colour phase
// is a product with two constant matrices formed at context creation
// (coarse_inverse):
//   x = A^-1 rhs = T - H X,  T = G S + g v_0,  G = (A^-1) rows 1.., H = qx G Bw
// with X the line's off-diagonal x terms (xoff), S its source, Bw the compact
// row weights and v_0 its wall value.  T does not change during the sweeps.
// What bounds the solve is the chain of 4 phases per sweep, not its bytes:
// the banded substitution (banbk5_poi) is 2 (ny - 1) dependent steps per
// phase whose factors come from scalar memory, about 60 cycles each; the
// product has none, runs on the matrix cores (v_mfma 16x16x4, both
// precisions) and needs one barrier per phase instead of two.  A workgroup
// takes one part (re or im: the operator is real) of one mode; a wavefront
// owns 16 lines of each colour, their v and T in registers in the result
// layout, and forms the operand X straight from the v columns in LDS; the two
// border lines are one further wavefront's scalar products.  Per call between
// events, banded substitution -> inverse form: FP64, 60 sweeps, 49x13x8 251 -> 70 us,
// 129x25x64 424 -> 160, 257x33x128 1774 -> 309, 129x24x20 (the lane scan) 1035
// -> 159; FP32, 5 sweeps, 129x25x64 32 -> 22.
// 16 NB rows and 4 KS columns hold the ny - 1 rows; THREADS bounds the
// registers (256 up to 144 columns: a wavefront may use the whole file).
typedef double mfma_d4 __attribute__((ext_vector_type(4)));
typedef float mfma_f4 __attribute__((ext_vector_type(4)));
template <typename T>
using Acc4 = std::conditional_t<sizeof(T) == 8, mfma_d4, mfma_f4>;
__device__ __forceinline__ mfma_d4 mfma4(double a, double b, mfma_d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mfma_f4 mfma4(float a, float b, mfma_f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// row of result element i of a lane (column lane % 16 in both layouts)
template <typename T>
__device__ __forceinline__ int acc_row(int lane, int i)
{
    return sizeof(T) == 8 ? 4 * i + lane / 16 : 4 * (lane / 16) + i;
}

template <typename T>
__host__ __device__ inline size_t coarse_inv_lds(int nx, int ny)
{
    return (static_cast<size_t>(coarse_stride(ny)) * nx + 64) * sizeof(T);
}

template <typename T, int KS, int THREADS>
__global__ void __launch_bounds__(THREADS) smooth_coarsest_inv_kernel(LevelArgs<T> L,
                                                                   cx<T> *__restrict__ V,
                                                                   const cx<T> *__restrict__ S,
                                                                   const T *__restrict__ inv,
                                                                   int sweeps, T rf,
                                                                   const int *active)
{
    constexpr int NB = (KS + 3) / 4, M = 16 * NB, N = 4 * KS;
    extern __shared__ unsigned char smem_raw[];
    const int k = blockIdx.x, part = blockIdx.y;
    if (active && !active[k]) return;
    const int nx = L.nx, ny = L.ny, ld = L.ld, LS = coarse_stride(ny);
    T *sv = reinterpret_cast<T *>(smem_raw);
    T *xb = sv + static_cast<size_t>(LS) * nx;       // the border lines' x terms
    T *gv = reinterpret_cast<T *>(V + static_cast<size_t>(k) * L.plane) + part;
    const T *gs = reinterpret_cast<const T *>(S + static_cast<size_t>(k) * L.plane) + part;
    const T *tab = inv + static_cast<size_t>(k) * 2 * coarse_inv_size(ny);
    for (int e = threadIdx.x; e < nx * ny; e += blockDim.x) {
        const int i = e / ny, j = e % ny;
        sv[i * LS + j] = gv[2 * (static_cast<size_t>(i) * ld + j)];
    }
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int n16 = lane % 16, q4 = lane / 16;
    const int waves = static_cast<int>(blockDim.x) / 64 - 1;   // and the border wavefront
    __syncthreads();
    if (wave == waves) {
        // the border lines: lane (line lane / M, row 1 + lane % M)
        const int line = lane / M, row = 1 + lane % M, rc = min(row, ny - 1);
        const bool own = line < 2 && row < ny;
        const int bc = line == 0 ? 1 : nx - 2, d = line == 0 ? LS : -LS;
        const T *bt = tab + coarse_inv_size(ny);
        const T *sc = gs + 2 * static_cast<size_t>(bc) * ld;
        T *c = sv + bc * LS + rc;
        T t = bt[rc - 1] * sv[bc * LS], v = *c, h[N];
        for (int j = 1; j < ny; ++j) t = fma(bt[M + (rc - 1) * N + j - 1], sc[2 * j], t);
#pragma unroll
        for (int j = 0; j < N; ++j) h[j] = bt[M + M * N + (rc - 1) * N + j];
        for (int it = 0; it < sweeps; ++it) {
            // rhs_border1/2: 10 a - 4 b + 14 c - 6 d + e
            if (line < 2)
                xb[lane] = fma(T(-6), c[3 * d], fma(T(14), c[2 * d], fma(T(-4), c[d], T(10) * c[-d])))
                           + c[4 * d];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (own) {
                T s0 = t, s1 = T(0), s2 = T(0), s3 = T(0);
#pragma unroll
                for (int j = 0; j < N; j += 4) {
                    const T *x = xb + line * M + j;
                    s0 = fma(-h[j], x[0], s0);
                    s1 = fma(-h[j + 1], x[1], s1);
                    s2 = fma(-h[j + 2], x[2], s2);
                    s3 = fma(-h[j + 3], x[3], s3);
                }
                v = fma(rf, ((s0 + s1) + (s2 + s3)) - v, v);
                *c = v;
            }
            for (int p = 0; p < 4; ++p) __syncthreads();
        }
    } else {
        // 16 lines of each colour; operand rows of this lane: row 1 + 4 s + q4
        // of k-step s (rows past ny read row ny - 1: their columns of G and H
        // are zero)
        const int n16 = lane % 16, q4 = lane / 16;
        T a[NB][KS];
        auto load_matrix = [&](const T *m) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int s = 0; s < KS; ++s) a[b][s] = m[(16 * b + n16) * N + 4 * s + q4];
        };
        int col[3];
        bool own[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const int c = 16 * wave + n16, nl = phase_lines(p + 1, nx);
            own[p] = c < nl;
            col[p] = phase_column(p + 1, min(c, nl - 1), nx);
        }
        // T = G S + g v_0, and the lines' own v
        T t[3][NB][4], v[3][NB][4];
        load_matrix(tab + M);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const T *sc = gs + 2 * static_cast<size_t>(col[p]) * ld;
            const T v0 = sv[col[p] * LS];
            T x[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) x[s] = sc[2 * min(1 + 4 * s + q4, ny - 1)];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                Acc4<T> acc;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = 16 * b + acc_row<T>(lane, i);
                    acc[i] = tab[r] * v0;
                    v[p][b][i] = sv[col[p] * LS + min(1 + r, ny - 1)];
                }
#pragma unroll
                for (int s = 0; s < KS; ++s) acc = mfma4(a[b][s], x[s], acc);
#pragma unroll
                for (int i = 0; i < 4; ++i) t[p][b][i] = acc[i];
            }
        }
        load_matrix(tab + M + M * N);
        // (the border wavefront may already have stored its first values: the
        // reads above are of this wavefront's own columns)
        for (int it = 0; it < sweeps; ++it) {
            __syncthreads();
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                T x[KS];
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const T *c = sv + col[p] * LS + min(1 + 4 * s + q4, ny - 1);
                    x[s] = fma(T(-16), c[-LS] + c[LS], c[-2 * LS] + c[2 * LS]);   // -X
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    Acc4<T> acc;
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = t[p][b][i];
#pragma unroll
                    for (int s = 0; s < KS; ++s) acc = mfma4(a[b][s], x[s], acc);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = 1 + 16 * b + acc_row<T>(lane, i);
                        v[p][b][i] = fma(rf, acc[i] - v[p][b][i], v[p][b][i]);
                        if (own[p] && r < ny) sv[col[p] * LS + r] = v[p][b][i];
                    }
                }
                __syncthreads();
            }
        }
    }
    for (int e = threadIdx.x; e < nx * ny; e += blockDim.x) {
        const int i = e / ny, j = e % ny;
        gv[2 * (static_cast<size_t>(i) * ld + j)] = sv[i * LS + j];
    }
}

// The tables of one line matrix (coarse_inv_size): a wavefront per matrix, a
// column of the inverse per lane, from the banded factors (l1, l2, u1, u2 and
// the pivot); then H = qx G Bw, where row j of Bw weighs the x terms of rows
// j-1, j, j+1 (rhs_center) and rows ny-2 and ny-1 take their own.
constexpr int kInvMaxNy = 33;
__global__ void __launch_bounds__(64) coarse_inverse_kernel(const double *__restrict__ lu, int lus,
                                                            int n, double sp1, double sp2,
                                                            double cp0, double cp1, double cp2,
                                                            double qx, double *__restrict__ inv,
                                                            float *__restrict__ invf)
{
    __shared__ double X[kInvMaxNy * kInvMaxNy];      // [row][column]
    const double *l1 = lu + static_cast<size_t>(blockIdx.x) * kLuFields * lus, *l2 = l1 + lus,
                 *u1 = l2 + lus, *u2 = u1 + lus, *pv = u2 + lus;
    const int c = threadIdx.x;
    if (c < n) {
        double a = 0.0, b = 0.0;
        for (int j = 0; j < n; ++j) {
            double x = j == c ? 1.0 : 0.0;
            if (j >= 1) x -= l1[j] * a;
            if (j >= 2) x -= l2[j] * b;
            X[j * n + c] = x;
            b = a;
            a = x;
        }
        a = b = 0.0;
        for (int j = n - 1; j >= 0; --j) {
            double x = X[j * n + c];
            if (j + 1 < n) x -= u1[j] * a;
            if (j + 2 < n) x -= u2[j] * b;
            x /= pv[j];
            X[j * n + c] = x;
            b = a;
            a = x;
        }
    }
    __syncthreads();
    const int cols = coarse_inv_cols(n), rows = coarse_inv_rows(n), size = rows * (1 + 2 * cols);
    for (int e = threadIdx.x; e < size; e += 64) {
        const int m = e < rows ? e : (e - rows) % (rows * cols);
        const int r = 1 + (e < rows ? m : m / cols), k = e < rows ? 0 : 1 + m % cols;
        double v = 0.0;
        if (r < n && k < n) {
            const double *x = X + r * n;
            if (e < rows + rows * cols) {
                v = x[k];
            } else {
                if (k == 1) v += sp1 * x[1];
                if (k == 2) v += sp2 * x[1];
                if (k >= 3 && k <= n - 2) v += cp2 * x[k - 1];
                if (k >= 2 && k <= n - 3) v += cp1 * x[k];
                if (k <= n - 4) v += cp0 * x[k + 1];
                if (k >= n - 2) v += x[k];
                v *= qx;
            }
        }
        const size_t o = static_cast<size_t>(blockIdx.x) * size + e;
        inv[o] = v;
        invf[o] = static_cast<float>(v);
    }
}

// k-steps of a level's row count
inline int coarse_inv_steps(int ny) { return std::max(2, (ny + 2) / 4); }
#define TBL_COARSE_KS(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8)

template <typename T, int G, int R>
static void launch_coarsest(const LevelArgs<T> &L, cx<T> *V, const cx<T> *S, const T *lu,
                            int sweeps, T rf, const int *active, hipStream_t st, int threads)
{
    const size_t shm = coarse_lds_bytes<T>(L.nx, L.ny, false);
    hipLaunchKernelGGL((smooth_coarsest_kernel<T, G, R>), dim3(L.K), dim3(threads), shm, st, L, V,
                       S, lu, sweeps, rf, active);
}

template <typename T>
int smooth_coarsest(const LevelArgs<T> &L, cx<T> *V, const cx<T> *S, const T *lu, const T *inv,
                    int sweeps, T rf, const int *active, int G, hipStream_t st)
{
    // shape kCoarseSeqShape: the inverse form where the context holds its
    // tables (coarse_inv_fits: faster at every size class of 33x9 to 257x33, six
    // FP64 sweeps 1.8 to 7.8 times, 33x33x16 29 against 54 us, 257x33x128 57 against
    // 163); any other shape, or a level it does not fit, the G-lane scan
    if (G == kCoarseSeqShape && inv) {
        const int ks = coarse_inv_steps(L.ny);
        const unsigned waves = static_cast<unsigned>((phase_lines(1, L.nx) + 15) / 16) + 1;
#define X(KS)                                                                                    \
    if (ks == KS) {                                                                              \
        const dim3 grid(L.K, 2), block(64 * waves);                                              \
        const size_t lds = coarse_inv_lds<T>(L.nx, L.ny);                                        \
        if (waves <= 4)                                                                          \
            hipLaunchKernelGGL((smooth_coarsest_inv_kernel<T, KS, 256>), grid, block, lds, st, L, \
                               V, S, inv, sweeps, rf, active);                                   \
        else if (waves <= 8)                                                                     \
            hipLaunchKernelGGL((smooth_coarsest_inv_kernel<T, KS, 512>), grid, block, lds, st, L, \
                               V, S, inv, sweeps, rf, active);                                   \
        else                                                                                     \
            hipLaunchKernelGGL((smooth_coarsest_inv_kernel<T, KS, 1024>), grid, block, lds, st,  \
                               L, V, S, inv, sweeps, rf, active);                                \
        return TBL_OK;                                                                           \
    }
        TBL_COARSE_KS(X)
#undef X
    }
    G = sweep_shape(G);
    if (coarse_lds_bytes<T>(L.nx, L.ny, false) > 160 * 1024)
        return smooth_sweeps<T>(L, V, S, lu, sweeps, rf, active,
                                shape_is_strip(G) ? G - kStripShape : G, nullptr, st);
    G = shape_lanes(G);
    const int R = line_rows_for(G, L.ny);
    if (R < 0) return TBL_ERR_GRID;
    bool done = false;
#define X(GG, RR)                                                                 \
    if (!done && G == GG && R == RR) {                                            \
        launch_coarsest<T, GG, RR>(L, V, S, lu, sweeps, rf, active, st, 512);     \
        done = true;                                                              \
    }
    TBL_LINE_SHAPES(X)
#undef X
    return done ? TBL_OK : TBL_ERR_GRID;
}

int coarse_kernel_attributes()
{
    hipError_t e = hipSuccess;
#define X(GG, RR)                                                                             \
    for (const void *f : {reinterpret_cast<const void *>(&smooth_coarsest_kernel<double, GG, RR>), \
                          reinterpret_cast<const void *>(&smooth_coarsest_kernel<float, GG, RR>)}) { \
        hipError_t r = allow_full_lds(f);                                                     \
        if (r != hipSuccess) e = r;                                                           \
    }
    TBL_LINE_SHAPES(X)
#undef X
#define X(KS)                                                                                   \
    for (const void *f :                                                                        \
         {reinterpret_cast<const void *>(&smooth_coarsest_inv_kernel<double, KS, 256>),         \
          reinterpret_cast<const void *>(&smooth_coarsest_inv_kernel<float, KS, 256>),          \
          reinterpret_cast<const void *>(&smooth_coarsest_inv_kernel<double, KS, 512>),         \
          reinterpret_cast<const void *>(&smooth_coarsest_inv_kernel<double, KS, 1024>),        \
          reinterpret_cast<const void *>(&smooth_coarsest_inv_kernel<float, KS, 512>),          \
          reinterpret_cast<const void *>(&smooth_coarsest_inv_kernel<float, KS, 1024>)}) {      \
        hipError_t r = allow_full_lds(f);                                                       \
        if (r != hipSuccess) e = r;                                                             \
    }
    TBL_COARSE_KS(X)
#undef X
    return e == hipSuccess ? TBL_OK : TBL_ERR_HIP;
}

// whether a level takes the inverse form: at most 32 rows besides the wall,
// 15 wavefronts of lines and the part's v in LDS
bool coarse_inv_fits(int nx, int ny)
{
    return ny <= kInvMaxNy && (phase_lines(1, nx) + 15) / 16 < 16 &&
           coarse_inv_lds<double>(nx, ny) <= 160 * 1024;
}

void coarse_inverse(const double *lu, int K, int ny, int lus, const double *sp, const double *cp,
                    double qx, double *inv, float *invf, hipStream_t st)
{
    hipLaunchKernelGGL(coarse_inverse_kernel, dim3(2 * K), dim3(64), 0, st, lu, lus, ny, sp[1], sp[2],
                       cp[0], cp[1], cp[2], qx, inv, invf);
}

template int smooth_coarsest<double>(const LevelArgs<double> &, cx<double> *, const cx<double> *,
                                     const double *, const double *, int, double, const int *, int,
                                     hipStream_t);
template int smooth_coarsest<float>(const LevelArgs<float> &, cx<float> *, const cx<float> *,
                                    const float *, const float *, int, float, const int *, int,
                                    hipStream_t);

}  // namespace tbl
