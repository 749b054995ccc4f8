// BF16 U-Net kernels for the learned multigrid initial guess (gfx950).
//
// Activations are NHWC (channels fastest).  3x3 convolutions run directly on the
// matrix cores (bf16 operands, fp32 accumulation), forward and backward, from
// input tiles in LDS; images too wide for those tiles take an im2col gather
// and a GEMM (weights: col^T x dZ, data: dZ x W^T and a col2im gather).
// Weights keep an fp32 master copy for Adam.
#include <algorithm>

#include "tbl_buf.h"
#include "tbl_nn.h"

namespace tbl {
namespace nn {

typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(bf16 h)
{
    return __uint_as_float(static_cast<unsigned>(h) << 16);
}

__device__ __forceinline__ bf16 f2bf(float f)
{
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return static_cast<bf16>((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
    u += 0x7fffu + ((u >> 16) & 1u);     // round to nearest even
    return static_cast<bf16>(u >> 16);
}

// ---------------------------------------------------------------------------
// GEMM  C[M,N] = alpha * A[M,K] B[K,N] + beta * C   (A, B bf16; C fp32)
// element (m,k) of A at A[m*sam + k*sak], (k,n) of B at B[k*sbk + n*sbn]
// Block: 256 threads = 4 wavefronts, tile 64 x 64, K step 32 through LDS;
// each wavefront owns a 32 x 32 sub-tile computed with 4 MFMAs per K step.
// ---------------------------------------------------------------------------
constexpr int BM = 64, BN = 64, BK = 32, PADK = BK + 4;

__global__ void __launch_bounds__(256) gemm_kernel(int M, int N, int K, const bf16 *A, long sam,
                                                   long sak, const bf16 *B, long sbk, long sbn,
                                                   float *C, long ldc, float alpha, float beta,
                                                   int kchunk)
{
    __shared__ bf16 As[BM][PADK];
    __shared__ bf16 Bs[BN][PADK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    float16v acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    const bool a_kfast = (sak == 1), b_kfast = (sbk == 1);
    const int kbeg = blockIdx.z * kchunk;
    const int kend = min(K, kbeg + kchunk);
    for (int k0 = kbeg; k0 < kend; k0 += BK) {
        // stage A (64 x 32) and B (32 x 64, stored transposed) in LDS
#pragma unroll
        for (int e = 0; e < (BM * BK) / 256; ++e) {
            const int idx = e * 256 + tid;
            int mm, kk;
            if (a_kfast) { mm = idx / BK; kk = idx % BK; }
            else         { kk = idx / BM; mm = idx % BM; }
            const int gm = m0 + mm, gk = k0 + kk;
            As[mm][kk] = (gm < M && gk < kend) ? A[gm * sam + gk * sak] : static_cast<bf16>(0);
        }
#pragma unroll
        for (int e = 0; e < (BN * BK) / 256; ++e) {
            const int idx = e * 256 + tid;
            int nn, kk;
            if (b_kfast) { nn = idx / BK; kk = idx % BK; }
            else         { kk = idx / BN; nn = idx % BN; }
            const int gn = n0 + nn, gk = k0 + kk;
            Bs[nn][kk] = (gn < N && gk < kend) ? B[gk * sbk + gn * sbn] : static_cast<bf16>(0);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BK; kk += 8) {
            const int kb = kk + (lane >> 5) * 4;
            short4v a, b;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                a[t] = static_cast<short>(As[wm + (lane & 31)][kb + t]);
                b[t] = static_cast<short>(Bs[wn + (lane & 31)][kb + t]);
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    // D layout: lane holds column (lane & 31); register i holds row
    // 8*(i/4) + 4*(lane/32) + (i%4)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = m0 + wm + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        const int col = n0 + wn + (lane & 31);
        if (row < M && col < N) {
            float *p = C + static_cast<long>(row) * ldc + col;
            const float v = alpha * acc[i];
            if (gridDim.z > 1) atomicAdd(p, v);
            else *p = (beta != 0.f) ? v + beta * *p : v;
        }
    }
}

__global__ void zero2d_kernel(int M, int N, float *C, long ldc)
{
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= static_cast<long>(M) * N) return;
    C[(e / N) * ldc + e % N] = 0.f;
}

// splitk > 1 partitions K over blockIdx.z and accumulates with atomics
// (C is cleared first; beta must be 0)
void gemm(int M, int N, int K, const bf16 *A, long sam, long sak, const bf16 *B, long sbk,
          long sbn, float *C, long ldc, float alpha, float beta, hipStream_t st, int splitk)
{
    if (splitk < 1) splitk = 1;
    int kchunk = (K + splitk - 1) / splitk;
    kchunk = (kchunk + BK - 1) / BK * BK;
    splitk = (K + kchunk - 1) / kchunk;
    if (splitk > 1) {
        const long mn = static_cast<long>(M) * N;
        hipLaunchKernelGGL(zero2d_kernel, dim3(static_cast<unsigned>((mn + 255) / 256)), dim3(256), 0,
                           st, M, N, C, ldc);
    }
    dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM, splitk);
    hipLaunchKernelGGL(gemm_kernel, grid, dim3(256), 0, st, M, N, K, A, sam, sak, B, sbk, sbn, C,
                       ldc, alpha, beta, kchunk);
}

// ---------------------------------------------------------------------------
// Direct 3x3 convolution (stride 1, zero padding 1) with bias and optional
// ReLU fused, bf16 NHWC in and out, for the forward pass.  The same product as
// im2col + GEMM (K index = tap * cin + c, taps row-major), without the
// im2col matrix or the fp32 pre-activation in HBM.
//
// Workgroup: 4 wavefronts; output tile = PX consecutive pixels of the
// flattened (image, row, column) index x CT output channels (CT = 64: 2x2
// wavefronts of 32x32; CT = 32: 4 wavefronts of 32 pixels), so narrow
// images fill whole tiles.  Per 32-channel input chunk the workgroup stages
// the chunk's packed weights [tap][cout][c] in LDS; each lane fetches its
// pixel's shifted input (4 channels, 8 bytes) straight from global memory
// (cached: neighbouring lanes and taps reuse the lines), and each wavefront
// runs 9 taps x 4 MFMAs (v_mfma_f32_32x32x8_bf16) per chunk.
// ---------------------------------------------------------------------------
constexpr int CK = 32;          // input channels per LDS chunk
constexpr int CKP = CK + 4;     // padded LDS row (bank spread)

// packed weights: wp[t][cout][cinp] (cinp = cin rounded up to CK, zero-filled)
__global__ void pack_conv3x3_kernel(int cin, int cinp, int cout, const bf16 *w, bf16 *wp)
{
    const long total = 9L * cout * cinp;
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    const int c = static_cast<int>(e % cinp);
    const int o = static_cast<int>((e / cinp) % cout);
    const int t = static_cast<int>(e / (static_cast<long>(cinp) * cout));
    wp[e] = (c < cin) ? w[(static_cast<long>(t) * cin + c) * cout + o] : static_cast<bf16>(0);
}

template <int CT>
__global__ void __launch_bounds__(256) conv3x3_kernel(long NP, int H, int W, int cin, int cinp,
                                                      int cout, const bf16 *__restrict__ X,
                                                      const bf16 *__restrict__ wp,
                                                      const float *__restrict__ bias,
                                                      bf16 *__restrict__ Y, int relu)
{
    constexpr int PX = (CT == 64) ? 64 : 128;
    __shared__ bf16 Ws[9][CT][CKP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long p0 = static_cast<long>(blockIdx.x) * PX;
    const int o0 = blockIdx.y * CT;
    const int wm = (CT == 64) ? (wave >> 1) * 32 : wave * 32;
    const int wn = (CT == 64) ? (wave & 1) * 32 : 0;
    // this lane's A-operand pixel (row of the 32x8 fragment)
    const long pa = p0 + wm + (lane & 31);
    const bool pa_ok = pa < NP;
    const int wa = static_cast<int>(pa % W), ha = static_cast<int>((pa / W) % H);
    const long na = pa / (static_cast<long>(W) * H);
    float16v acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    for (int c0 = 0; c0 < cinp; c0 += CK) {
        // weights of this chunk: [tap][cout o0..o0+CT][c0..c0+CK]
        for (int e = tid; e < 9 * CT * (CK / 4); e += 256) {
            const int q = e % (CK / 4), o = (e / (CK / 4)) % CT, t = e / ((CK / 4) * CT);
            *reinterpret_cast<short4v *>(&Ws[t][o][4 * q]) = *reinterpret_cast<const short4v *>(
                wp + (static_cast<long>(t) * cout + o0 + o) * cinp + c0 + 4 * q);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int hh = ha + t / 3 - 1, ww = wa + t % 3 - 1;
            const bool ok = pa_ok && hh >= 0 && hh < H && ww >= 0 && ww < W;
            const bf16 *src = X + ((na * H + hh) * W + ww) * cin;
#pragma unroll
            for (int kk = 0; kk < CK; kk += 8) {
                const int kb = kk + (lane >> 5) * 4;
                // cin is a multiple of 4: the 4 channels are all in range or none
                short4v a = {0, 0, 0, 0};
                if (ok && c0 + kb < cin) a = *reinterpret_cast<const short4v *>(src + c0 + kb);
                const short4v b = *reinterpret_cast<const short4v *>(&Ws[t][wn + (lane & 31)][kb]);
                acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // D layout: lane holds output channel (lane & 31); register i holds pixel
    // 8*(i/4) + 4*(lane/32) + (i%4) of the wavefront's 32
    const int o = o0 + wn + (lane & 31);
    const float bo = bias[o];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const long p = p0 + wm + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (p < NP) {
            float v = acc[i] + bo;
            if (relu) v = fmaxf(v, 0.f);
            Y[p * cout + o] = f2bf(v);
        }
    }
}

// Same convolution with the input staged in LDS, on gfx950's K=16 matrix
// instruction (v_mfma_f32_32x32x16_bf16): a workgroup owns PX consecutive
// flattened output pixels (4 wavefronts x MT 32-pixel tiles) and CT = 32
// output channels.  Per 32-channel chunk it holds the packed weights and the
// PX + 2W + 2 input pixels its 3x3 taps can reach in LDS.  The next chunk's
// global loads (NI 16-byte pieces of input and the weights per thread) are
// issued before the current chunk's arithmetic and written to LDS after it.
// The weights are the first operand, the pixels the second: a lane's results
// are 4 consecutive channels of one pixel, 8-byte stores.
//
// What bounds it: LDS reads (3 fragments of 1 KB for 2 MFMAs with MT = 2, 128 B
// a clock) and the loads' latency, one per chunk: three workgroups a CU cover
// more of it than twice the channels each (a quarter slower) or a loop over
// tiles with the next one's loads ahead (the registers).  So rows are
// 64 bytes with their pieces permuted against bank conflicts (not padded to
// 80), offsets are 32-bit and formed once, and a tap outside the image reads a
// row of zeros instead of branching.  Four input channels (CIN4: the first
// layer) take one 8-byte piece a pixel and the first half of a chunk's K; the
// other half would add zeros.  64 images of
// 32x136, the 14 layers together: 448 -> 243 us (with padded rows, branches,
// 64-bit divisions and 2-byte stores: 2.1 to 1.2 times each).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// byte offset of piece p (8 channels) of row r in LDS.  A 16-byte LDS access
// takes 16 lanes at a time, 0-3, 12-15, 20-27 (and 4-11, 16-19, 28-31, and so in
// the upper half): a piece of these rows after any first row, and the pieces of
// 4 rows, lie in 16 different columns of the 256 bytes.
__device__ __forceinline__ unsigned conv_slot(unsigned r, unsigned p)
{
    return r * 64 + ((p ^ (r >> 2 & 3)) << 4);
}

template <int MT, int NI, bool CIN4>
__global__ void __launch_bounds__(256, 3) conv3x3s_kernel(int NP, int H, int W, int cin, int cinp,
                                                       int cout, const bf16 *__restrict__ X,
                                                       const bf16 *__restrict__ wp,
                                                       const float *__restrict__ bias,
                                                       bf16 *__restrict__ Y, int relu)
{
    constexpr int CT = 32, PX = 128 * MT, WPT = (9 * CT * 4 + 255) / 256;
    extern __shared__ __attribute__((aligned(16))) unsigned char conv_smem[];
    unsigned char *Ws = conv_smem, *Xs = Ws + 9 * CT * 64;
    const int NQ = PX + 2 * W + 2;                // staged pixels; row NQ: zeros
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
    const int p0 = static_cast<int>(blockIdx.x) * PX;
    const int q0 = p0 - W - 1;                    // pixel of Xs row 0
    const int o0 = blockIdx.y * CT;
    // buffer resources: the weights, and the activations from the tile's
    // first reachable pixel; pieces outside the batch read zero
    const int qb = q0 > 0 ? q0 : 0;
    const __amdgpu_buffer_rsrc_t wres =
        buf_rsrc_uniform(wp, static_cast<size_t>(9) * cout * cinp * sizeof(bf16));
    const __amdgpu_buffer_rsrc_t xres = buf_rsrc_uniform(
        X + static_cast<size_t>(qb) * cin,
        static_cast<size_t>(min(NP - qb, NQ)) * cin * sizeof(bf16));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    // this thread's first pieces; the others follow at uniform distances (64 rows
    // of weights, or 64 pixels, 256 with CIN4), past the last one past the range;
    // before the batch (the first tile) the offset wraps past it
    const unsigned wo = static_cast<unsigned>(((tid / 4 / CT * cout + o0 + tid / 4 % CT) * cinp + 8 * (tid % 4)) * 2);
    const unsigned wd = static_cast<unsigned>((64 / CT) * cout * cinp * 2);
    const unsigned xo = static_cast<unsigned>(
        (q0 - qb) * cin * 2 + (CIN4 ? tid * cin * 2 : (tid / 4 * cin + 8 * (tid % 4)) * 2));
    const unsigned xd = static_cast<unsigned>((CIN4 ? 256 : 64) * cin * 2);
    u4 wr[WPT], xr[NI];
    auto fetch = [&](int c0) {
#pragma unroll
        for (int s = 0; s < WPT; ++s)
            wr[s] = __builtin_amdgcn_raw_buffer_load_b128(wres, wo + (s * wd + 2 * c0), 0, 0);
#pragma unroll
        for (int s = 0; s < NI; ++s) {
            if constexpr (CIN4) {
                const u2 v = __builtin_amdgcn_raw_buffer_load_b64(xres, xo + s * xd, 0, 0);
                xr[s] = u4{v.x, v.y, 0, 0};
            } else {
                xr[s] = __builtin_amdgcn_raw_buffer_load_b128(xres, xo + (s * xd + 2 * c0), 0, 0);
            }
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int s = 0; s < WPT; ++s) {
            const int e = tid + 256 * s;
            if (256 * (s + 1) <= 9 * CT * 4 || e < 9 * CT * 4)
                *reinterpret_cast<u4 *>(Ws + conv_slot(e / 4, e % 4)) = wr[s];
        }
#pragma unroll
        for (int s = 0; s < NI; ++s) {
            const int e = tid + 256 * s, q = CIN4 ? e : e / 4, g = CIN4 ? 0 : e % 4;
            if (q < NQ) *reinterpret_cast<u4 *>(Xs + conv_slot(q, g)) = xr[s];
        }
    };
    fetch(0);
    if (tid < 4) *reinterpret_cast<u4 *>(Xs + NQ * 64 + 16 * tid) = u4{0, 0, 0, 0};
    // this lane's pixels: offsets of their fragments per tap (K 8 half .. + 7)
    unsigned xa[MT][9];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int lp = wave * 32 * MT + m * 32 + (lane & 31);
        const unsigned pa = static_cast<unsigned>(p0 + lp), row = pa / static_cast<unsigned>(W);
        const int wa = static_cast<int>(pa - row * W), ha = static_cast<int>(row % static_cast<unsigned>(H));
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int hh = ha + t / 3 - 1, ww = wa + t % 3 - 1;
            const bool ok = (static_cast<unsigned>(hh) < static_cast<unsigned>(H)) &
                            (static_cast<unsigned>(ww) < static_cast<unsigned>(W)) &
                            (!CIN4 || half == 0);
            const unsigned r = static_cast<unsigned>(lp + W + 1 + (t / 3 - 1) * W + t % 3 - 1);
            xa[m][t] = ok ? conv_slot(r, half) : static_cast<unsigned>(NQ * 64);
        }
    }
    const unsigned wa0 = conv_slot(lane & 31, half);   // + 64 bytes per further row
    float16v acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[m][i] = 0.f;
    stash();
    __syncthreads();
    for (int c0 = 0; c0 < cinp; c0 += CK) {
        const bool more = c0 + CK < cinp;
        if (more) fetch(c0 + CK);
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int kk = 0; kk < (CIN4 ? 1 : 2); ++kk) {     // pieces half + 2 kk
                const bf16x8 b = *reinterpret_cast<const bf16x8 *>(Ws + t * CT * 64 + (wa0 ^ (32 * kk)));
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const bf16x8 a = *reinterpret_cast<const bf16x8 *>(Xs + (xa[m][t] ^ (32 * kk)));
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, acc[m], 0, 0, 0);
                }
            }
        __syncthreads();
        if (more) {
            stash();
            __syncthreads();
        }
    }
    // D layout: lane holds pixel (lane & 31); register i output channel
    // 8*(i/4) + 4*half + (i%4) of the 32
    const int o = o0 + 4 * half;
    f32x4 bo[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) bo[g] = *reinterpret_cast<const f32x4 *>(bias + o + 8 * g);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p = p0 + wave * 32 * MT + m * 32 + (lane & 31);
        if (p >= NP) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = acc[m][4 * g + i] + bo[g][i];
                if (relu) v[i] = fmaxf(v[i], 0.f);
            }
            u2 y;
            y.x = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{v[0], v[1]}), bf16x2));
            y.y = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{v[2], v[3]}), bf16x2));
            *reinterpret_cast<u2 *>(Y + static_cast<size_t>(p) * cout + o + 8 * g) = y;
        }
    }
}

// ---------------------------------------------------------------------------
// Backward of a 3x3 convolution without the im2col and col2im matrices (9
// times the activations, bf16 and fp32, each written and read once), which
// with the GEMM's scalar loads were the time of a training step.
//
// Gradient of the input: dX[p, ci] = sum_t sum_co dZ[p - shift(t), co] W[t, ci,
// co].  Workgroup: 4 wavefronts x MT tiles of 32 flattened pixels x CT = 32 NT
// input channels; LDS: the dZ pixels its taps reach, all COUT channels, and
// one tap's weights (the next tap's loads are in flight meanwhile; the bf16
// weights [tap][ci][co] need no packing).  Each tap is summed over the channels on
// its own and the taps are added in fp32 in their order, as the GEMM and
// col2im did: the same values bit for bit (the K = 16 instruction adds as two
// of K = 8 do), so no bf16 rounding downstream changes.
// ---------------------------------------------------------------------------
template <int MT, int NT, int COUT>
__global__ void __launch_bounds__(256) conv3x3_dx_kernel(long NP, int H, int W, int cin,
                                                         const bf16 *__restrict__ dZ,
                                                         const bf16 *__restrict__ wb,
                                                         float *__restrict__ dX)
{
    constexpr int CT = 32 * NT, PX = 128 * MT, ROW = COUT + 8, G = COUT / 8;
    constexpr int WP = CT * G / 256 > 0 ? CT * G / 256 : 1;
    extern __shared__ __attribute__((aligned(16))) unsigned char conv_smem[];
    bf16 *Ws = reinterpret_cast<bf16 *>(conv_smem), *Zs = Ws + CT * ROW;
    const int NQ = PX + 2 * W + 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long p0 = static_cast<long>(blockIdx.x) * PX, q0 = p0 - W - 1;
    const int o0 = blockIdx.y * CT;
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    // weights of tap t, rows o0 .. (zero past cin)
    u4 wr[WP];
    auto fetch = [&](int t) {
#pragma unroll
        for (int s = 0; s < WP; ++s) {
            const int e = tid + 256 * s, o = e / G, g = e % G;
            wr[s] = u4{0, 0, 0, 0};
            if (e < CT * G && o0 + o < cin)
                wr[s] = *reinterpret_cast<const u4 *>(
                    wb + (static_cast<long>(t) * cin + o0 + o) * COUT + 8 * g);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int s = 0; s < WP; ++s) {
            const int e = tid + 256 * s;
            if (e < CT * G) *reinterpret_cast<u4 *>(Ws + e / G * ROW + 8 * (e % G)) = wr[s];
        }
    };
    fetch(0);
    for (int e = tid; e < NQ * G; e += 256) {
        const int q = e / G, g = e % G;
        const long gp = q0 + q;
        u4 v = {0, 0, 0, 0};
        if (gp >= 0 && gp < NP) v = *reinterpret_cast<const u4 *>(dZ + gp * COUT + 8 * g);
        *reinterpret_cast<u4 *>(Zs + q * ROW + 8 * g) = v;
    }
    stash();
    int lq[MT];
    unsigned tapok[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int lp = wave * 32 * MT + m * 32 + (lane & 31);
        const long pa = p0 + lp;
        const int wa = static_cast<int>(pa % W), ha = static_cast<int>((pa / W) % H);
        unsigned ok = 0;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int hh = ha - (t / 3 - 1), ww = wa - (t % 3 - 1);
            if (pa < NP && hh >= 0 && hh < H && ww >= 0 && ww < W) ok |= 1u << t;
        }
        lq[m] = lp + W + 1;
        tapok[m] = ok;
    }
    float16v sum[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[m][n][i] = 0.f;
    __syncthreads();
#pragma unroll 1
    for (int t = 0; t < 9; ++t) {
        if (t < 8) fetch(t + 1);
        const int sh = (t / 3 - 1) * W + (t % 3 - 1);
        float16v acc[MT][NT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[m][n][i] = 0.f;
#pragma unroll 4
        for (int kk = 0; kk < COUT; kk += 16) {
            const int kb = kk + (lane >> 5) * 8;
            bf16x8 b[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n)
                b[n] = *reinterpret_cast<const bf16x8 *>(Ws + (n * 32 + (lane & 31)) * ROW + kb);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                bf16x8 a = {};
                if (tapok[m] >> t & 1u)
                    a = *reinterpret_cast<const bf16x8 *>(Zs + (lq[m] - sh) * ROW + kb);
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[n], acc[m][n], 0, 0, 0);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) sum[m][n][i] += acc[m][n][i];
        __syncthreads();
        if (t < 8) {
            stash();
            __syncthreads();
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int o = o0 + n * 32 + (lane & 31);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const long p = p0 + wave * 32 * MT + m * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                if (p < NP && o < cin) dX[p * cin + o] = sum[m][n][i];
            }
    }
}

// Gradient of the weights: dW[t, ci, co] = sum_p X[p + shift(t), ci] dZ[p, co].
// Workgroup: 32 input channels x 32 NC output channels x all 9 taps over a
// range of row groups; its wavefronts take NC channel blocks x 4 / NC shares
// of the taps.  Per group of nr image rows LDS holds the input rows -1 ..
// nr, a zero column each side and one zero row (for the taps outside the
// image), and the dZ pixels, both as they lie in memory: 16 channel pairs of
// 4 bytes per pixel and 8 bytes of padding, so a lane's pair of one pixel is one
// 4-byte read, the four pixel groups of a wavefront fall on different banks,
// and a tap is a constant offset from the pixel's address.  Eight pixels of a
// pair are turned into two operands (the even and the odd channel of 8
// pixels) by byte permutes: 4 MFMAs 16x16x32 per tap and 8 reads.  Partial
// sums go to a workspace, one slice per blockIdx.x, and are added in order
// by wgrad_reduce_kernel: no atomics, the same bits every run.
constexpr int kWgRow = 36;                     // bf16 per staged pixel
// bytes of the staged input rows, a multiple of 16
__host__ __device__ inline size_t dw_x_bytes(int nr, int w)
{
    return (static_cast<size_t>(nr + 3) * (w + 2) * kWgRow * sizeof(bf16) + 15) / 16 * 16;
}

template <int NC>
__global__ void __launch_bounds__(256) conv3x3_dw_kernel(int rows, int H, int W, int nr, int ks,
                                                         int cin, int cout,
                                                         const bf16 *__restrict__ X,
                                                         const bf16 *__restrict__ dZ,
                                                         float *__restrict__ ws)
{
    constexpr int KW = 4 / NC, TM = (8 + KW) / KW;
    extern __shared__ __attribute__((aligned(16))) unsigned char conv_smem[];
    const int W2 = W + 2, np = 32 * ks;        // padded row, pixels of a group
    bf16 *Xs = reinterpret_cast<bf16 *>(conv_smem);
    bf16 *Zs = Xs + dw_x_bytes(nr, W) / sizeof(bf16);   // [NC][np]
    uint16_t *at = reinterpret_cast<uint16_t *>(Zs + NC * np * kWgRow);   // [3][np]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nc = wave % NC, kw = __builtin_amdgcn_readfirstlane(wave / NC);
    const int c0 = blockIdx.y * 32, o0 = blockIdx.z * 32 * NC;
    const int m4 = (lane & 15) * 4, g = lane >> 4;
    // the zero borders, written once
    for (int e = tid; e < (nr + 3) * W2 * (kWgRow / 4); e += 256) {
        const int q = e / (kWgRow / 4), col = q % W2;
        if (col == 0 || col == W + 1 || q / W2 == nr + 2)
            *reinterpret_cast<short4v *>(Xs + q * kWgRow + 4 * (e % (kWgRow / 4))) = short4v{0, 0, 0, 0};
    }
    f32x4 acc[TM][2][2];
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e >> 1][e & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __amdgpu_buffer_rsrc_t xr =
        buf_rsrc_uniform(X, static_cast<size_t>(rows) * W * cin * sizeof(bf16));
    const __amdgpu_buffer_rsrc_t zr =
        buf_rsrc_uniform(dZ, static_cast<size_t>(rows) * W * cout * sizeof(bf16));
    const int groups = (rows + nr - 1) / nr;
    for (int grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const int r0 = grp * nr;
        __syncthreads();
        // input rows r0 - 1 .. r0 + nr (rows of all images are contiguous; past
        // either end the buffer reads zero), 8 or (cin 4) 4 channels a piece,
        // the loads of NI pieces in flight together
        constexpr int NI = 6;
        if (cin >= 8) {
            const int n = (nr + 2) * W, dq = 64 / W, dr = 64 % W, cg = (tid & 3) * 8;
            int q = tid >> 2, lr = q / W, col = q % W;
            while (q < n) {
                u32x4 v[NI];
                int at_[NI];
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const unsigned off = static_cast<unsigned>((((r0 - 1) * W + q) * cin + c0 + cg) * 2);
                    v[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, q < n && c0 + cg < cin ? off : kBufOff, 0, 0);
                    at_[i] = q < n ? q + 2 * lr + 1 : -1;
                    q += 64;
                    lr += dq;
                    col += dr;
                    if (col >= W) {
                        col -= W;
                        ++lr;
                    }
                }
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    if (at_[i] >= 0) {
                        u32x2 *d = reinterpret_cast<u32x2 *>(Xs + at_[i] * kWgRow + cg);
                        d[0] = u32x2{v[i][0], v[i][1]};
                        d[1] = u32x2{v[i][2], v[i][3]};
                    }
            }
        } else {
            for (int q = tid; q < (nr + 2) * W; q += 256) {
                const unsigned off = static_cast<unsigned>(((r0 - 1) * W + q) * cin * 2);
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(xr, off, 0, 0);
                bf16 *d = Xs + (q + 2 * (q / W) + 1) * kWgRow;
#pragma unroll
                for (int c = 0; c < 32; c += 4) *reinterpret_cast<u32x2 *>(d + c) = c ? u32x2{0, 0} : v;
            }
        }
        {
            const int n = np * NC * 4;
            for (int e0 = tid; e0 < n; e0 += 256 * NI) {
                u32x4 v[NI];
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int e = e0 + 256 * i, p = e / (4 * NC), c = e % (4 * NC) * 8;
                    const unsigned off = static_cast<unsigned>(((r0 * W + p) * cout + o0 + c) * 2);
                    v[i] = __builtin_amdgcn_raw_buffer_load_b128(zr, p < nr * W ? off : kBufOff, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int e = e0 + 256 * i, p = e / (4 * NC), c = e % (4 * NC) * 8;
                    if (e < n) {
                        u32x2 *d = reinterpret_cast<u32x2 *>(Zs + (c / 32 * np + p) * kWgRow + c % 32);
                        d[0] = u32x2{v[i][0], v[i][1]};
                        d[1] = u32x2{v[i][2], v[i][3]};
                    }
                }
            }
        }
        // staged row of each pixel for the three tap rows, in units of 8 bytes
        for (int p = tid; p < np; p += 256) {
            const int lr = p / W, col = p % W, h = (r0 + lr) % H;
            const bool in = p < nr * W;
#pragma unroll
            for (int dh = -1; dh <= 1; ++dh) {
                const int row = in && h + dh >= 0 && h + dh < H ? lr + 1 + dh : nr + 2;
                at[(dh + 1) * np + p] =
                    static_cast<uint16_t>((row * W2 + (in ? col : 0) + 1) * (kWgRow / 4));
            }
        }
        __syncthreads();
        for (int k = 0; k < ks; ++k) {
            auto pairs = [&](const unsigned (&w)[8], bf16x8 &even, bf16x8 &odd) {
                unsigned ev[4], od[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    ev[i] = __builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], 0x05040100u);
                    od[i] = __builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], 0x07060302u);
                }
                __builtin_memcpy(&even, ev, 16);
                __builtin_memcpy(&odd, od, 16);
            };
            bf16x8 b[2];
            {
                unsigned w[8];
                const unsigned char *z = reinterpret_cast<const unsigned char *>(
                                             Zs + (nc * np + 32 * k + 8 * g) * kWgRow) + m4;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    w[j] = *reinterpret_cast<const unsigned *>(z + j * kWgRow * 2);
                pairs(w, b[0], b[1]);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int t = kw + KW * i;
                if (t < 9) {
                    uint16_t a8[8];
                    __builtin_memcpy(a8, __builtin_assume_aligned(at + t / 3 * np + 32 * k + 8 * g, 16), 16);
                    const unsigned char *x = conv_smem + m4 + (t % 3 - 1) * kWgRow * 2;
                    unsigned w[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) w[j] = *reinterpret_cast<const unsigned *>(x + 8 * a8[j]);
                    bf16x8 a[2];
                    pairs(w, a[0], a[1]);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[i][e >> 1][e & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            a[e >> 1], b[e & 1], acc[i][e >> 1][e & 1], 0, 0, 0);
                }
            }
        }
    }
    float *out = ws + static_cast<size_t>(blockIdx.x) * 9 * cin * cout;
#pragma unroll
    for (int q = 0; q < TM; ++q)
#pragma unroll
        for (int ea = 0; ea < 2; ++ea)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = kw + KW * q, c = c0 + 2 * (4 * g + i) + ea;
                if (t < 9 && c < cin)
                    *reinterpret_cast<float2 *>(
                        out + (static_cast<size_t>(t) * cin + c) * cout + o0 + 32 * nc + (lane & 15) * 2) =
                        float2{acc[q][ea][0][i], acc[q][ea][1][i]};
            }
}

// g[e] = sum over the slices of ws, the bias partials bs likewise: 64 sums per
// workgroup, four shares of the slices each, added in order
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(int n, int slices,
                                                           const float *__restrict__ ws,
                                                           float *__restrict__ g, int cout, int bslices,
                                                           const float *__restrict__ bs,
                                                           float *__restrict__ gb)
{
    __shared__ float part[256];
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;
    const bool w = e < n;
    const float *src = w ? ws + e : bs + (e - n);
    const int m = w ? slices : bslices, per = (m + 3) / 4, stride = w ? n : cout;
    float s = 0.f;
    if (e < n + cout) {
        const int m1 = min(m, (q + 1) * per);
#pragma unroll 8
        for (int k = q * per; k < m1; ++k) s += src[static_cast<size_t>(k) * stride];
    }
    part[threadIdx.x] = s;
    __syncthreads();
    if (q == 0 && e < n + cout)
        (w ? g[e] : gb[e - n]) = ((s + part[threadIdx.x + 64]) + part[threadIdx.x + 128]) + part[threadIdx.x + 192];
}

// dZ = dY * (y > 0) as bf16, and the block's sums of dZ per channel
// (bs[block][Cc]): four channels per thread, Cc / 4 threads a pixel; Cc a
// multiple of 4 that divides 1024
__global__ void __launch_bounds__(256) relu_back_bias_kernel(long P, int Cc, long per,
                                                             const float *__restrict__ dY,
                                                             const bf16 *__restrict__ y,
                                                             bf16 *__restrict__ dZ,
                                                             float *__restrict__ bs)
{
    __shared__ float red[256][4];
    const int cg = Cc / 4, c = (threadIdx.x % cg) * 4, px = threadIdx.x / cg, step = 256 / cg;
    const long p1 = min(P, (blockIdx.x + 1) * per);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (long p = blockIdx.x * per + px; p < p1; p += step) {
        const float4 d = *reinterpret_cast<const float4 *>(dY + p * Cc + c);
        const short4v a = *reinterpret_cast<const short4v *>(y + p * Cc + c);
        const float v[4] = {d.x, d.y, d.z, d.w};
        short4v z;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bf16 b = f2bf(bf2f(static_cast<bf16>(a[q])) > 0.f ? v[q] : 0.f);
            z[q] = static_cast<short>(b);
            s[q] += bf2f(b);
        }
        *reinterpret_cast<short4v *>(dZ + p * Cc + c) = z;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) red[threadIdx.x][q] = s[q];
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < Cc) {
        float t = 0.f;
        for (int q = 0; q < step; ++q) t += red[q * cg + threadIdx.x / 4][threadIdx.x % 4];
        bs[static_cast<size_t>(blockIdx.x) * Cc + threadIdx.x] = t;
    }
}

// Backward of the 1x1 output layer (cin inputs of 32, two outputs): dX = dZ W^T,
// and the block's sums of X^T dZ and dZ.  One input channel and pixel per thread.
__global__ void __launch_bounds__(256) out_back_kernel(long P, long per, const float *__restrict__ dY,
                                                       const bf16 *__restrict__ X,
                                                       const bf16 *__restrict__ w,
                                                       float *__restrict__ dX,
                                                       float *__restrict__ ws, float *__restrict__ bs)
{
    __shared__ float red[256][4];
    const int c = threadIdx.x & 31, px = threadIdx.x >> 5;
    const float w0 = bf2f(w[2 * c]), w1 = bf2f(w[2 * c + 1]);
    const long p1 = min(P, (blockIdx.x + 1) * per);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (long p = blockIdx.x * per + px; p < p1; p += 8) {
        const float2 d = *reinterpret_cast<const float2 *>(dY + 2 * p);
        const float z0 = bf2f(f2bf(d.x)), z1 = bf2f(f2bf(d.y)), x = bf2f(X[32 * p + c]);
        dX[32 * p + c] = __builtin_fmaf(z1, w1, z0 * w0);
        s[0] += x * z0;
        s[1] += x * z1;
        s[2] += z0;
        s[3] += z1;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) red[threadIdx.x][q] = s[q];
    __syncthreads();
    if (threadIdx.x < 64) {
        float t = 0.f;
        for (int q = 0; q < 8; ++q) t += red[32 * q + threadIdx.x / 2][threadIdx.x % 2];
        ws[blockIdx.x * 64 + threadIdx.x] = t;
    } else if (threadIdx.x < 66) {
        float t = 0.f;
        for (int q = 0; q < 8; ++q) t += red[32 * q][2 + threadIdx.x - 64];
        bs[blockIdx.x * 2 + threadIdx.x - 64] = t;
    }
}

// ---------------------------------------------------------------------------
// element-wise and layout kernels
// ---------------------------------------------------------------------------
static inline unsigned nb(long n) { return static_cast<unsigned>((n + 255) / 256); }

// col[p, t*C + c] = X[n, h+dh, w+dw, c] (zero outside), taps t = (dh+1)*3 + (dw+1)
__global__ void im2col_kernel(int Nn, int H, int W, int Cc, const bf16 *X, bf16 *col)
{
    const long total = static_cast<long>(Nn) * H * W * 9 * Cc;
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    const int c = static_cast<int>(e % Cc);
    long r = e / Cc;
    const int t = static_cast<int>(r % 9);
    const long p = r / 9;
    const int w = static_cast<int>(p % W), h = static_cast<int>((p / W) % H);
    const int n = static_cast<int>(p / (static_cast<long>(W) * H));
    const int hh = h + t / 3 - 1, ww = w + t % 3 - 1;
    bf16 v = 0;
    if (hh >= 0 && hh < H && ww >= 0 && ww < W)
        v = X[((static_cast<long>(n) * H + hh) * W + ww) * Cc + c];
    col[e] = v;
}

// dX[n,h,w,c] = sum_t dcol[(n, h-dh, w-dw), t*C + c]
__global__ void col2im_kernel(int Nn, int H, int W, int Cc, const float *dcol, float *dX, int accumulate)
{
    const long total = static_cast<long>(Nn) * H * W * Cc;
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    const int c = static_cast<int>(e % Cc);
    const long p = e / Cc;
    const int w = static_cast<int>(p % W), h = static_cast<int>((p / W) % H);
    const int n = static_cast<int>(p / (static_cast<long>(W) * H));
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        const int hh = h - (t / 3 - 1), ww = w - (t % 3 - 1);
        if (hh >= 0 && hh < H && ww >= 0 && ww < W)
            s += dcol[(((static_cast<long>(n) * H + hh) * W + ww) * 9 + t) * Cc + c];
    }
    dX[e] = accumulate ? dX[e] + s : s;
}

// The output layer, 1x1 from 32 channels to 2, with bias: four lanes a pixel, 8
// channels (16 bytes) each, fp32 sums.  A 64-wide GEMM tile has no use for two
// columns, and its bias took a pass of its own: 64 images of 32x136 (20 MB)
// 32 -> 5.6 us.
__global__ void __launch_bounds__(256) out_kernel(unsigned P, const bf16 *__restrict__ x,
                                                  const bf16 *__restrict__ w,
                                                  const float *__restrict__ b, float *__restrict__ y)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const unsigned e = blockIdx.x * 256u + threadIdx.x, p = e / 4, q = e % 4;
    if (p >= P) return;
    const u4 v = *reinterpret_cast<const u4 *>(x + static_cast<size_t>(p) * 32 + 8 * q);
    const u4 w0 = reinterpret_cast<const u4 *>(w)[2 * q], w1 = reinterpret_cast<const u4 *>(w)[2 * q + 1];
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const unsigned t = v[c / 2], u = c < 4 ? w0[c] : w1[c - 4];      // w[channel][output]
        const float a = __uint_as_float(c % 2 ? t & 0xffff0000u : t << 16);
        s0 = fmaf(a, __uint_as_float(u << 16), s0);
        s1 = fmaf(a, __uint_as_float(u & 0xffff0000u), s1);
    }
    s0 += __shfl_xor(s0, 1, 4);
    s1 += __shfl_xor(s1, 1, 4);
    s0 += __shfl_xor(s0, 2, 4);
    s1 += __shfl_xor(s1, 2, 4);
    if (q < 2) y[2 * static_cast<size_t>(p) + q] = (q ? s1 : s0) + b[q];
}

__global__ void relu_back_kernel(long n, const float *dY, const bf16 *y, bf16 *dZ, int relu)
{
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= n) return;
    float g = dY[e];
    if (relu && !(bf2f(y[e]) > 0.f)) g = 0.f;
    dZ[e] = f2bf(g);
}

// db[c] = sum_p dZ[p, c]
__global__ void bias_grad_kernel(long P, int Cc, const bf16 *dZ, float *db)
{
    const int c = blockIdx.x;
    float s = 0.f;
    for (long p = threadIdx.x; p < P; p += 256) s += bf2f(dZ[p * Cc + c]);
    __shared__ float red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[c] = red[0];
}

// 2x2 average pooling, NHWC, 8 channels a thread (total: outputs / 8)
__global__ void __launch_bounds__(256) pool_kernel(unsigned total, unsigned H2, unsigned W2, unsigned G,
                                                   const bf16 *__restrict__ X, bf16 *__restrict__ Y)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const unsigned e = blockIdx.x * 256u + threadIdx.x;
    if (e >= total) return;
    const unsigned p = e / G, g = e % G, r = p / W2, w = p % W2;         // r: image and row
    const u4 *x = reinterpret_cast<const u4 *>(X) + ((static_cast<size_t>(2) * r * 2 * W2 + 2 * w) * G + g);
    const u4 a = x[0], b = x[G], c = x[static_cast<size_t>(2) * W2 * G], d = x[(static_cast<size_t>(2) * W2 + 1) * G];
    u4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        auto lo = [](unsigned v) { return __uint_as_float(v << 16); };
        auto hi = [](unsigned v) { return __uint_as_float(v & 0xffff0000u); };
        const unsigned l = f2bf(0.25f * (lo(a[i]) + lo(b[i]) + lo(c[i]) + lo(d[i])));
        y[i] = l | static_cast<unsigned>(f2bf(0.25f * (hi(a[i]) + hi(b[i]) + hi(c[i]) + hi(d[i])))) << 16;
    }
    reinterpret_cast<u4 *>(Y)[e] = y;
}

__global__ void pool_back_kernel(int Nn, int H, int W, int Cc, const float *dY, float *dX, int accumulate)
{
    const long total = static_cast<long>(Nn) * H * W * Cc;
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    const int c = static_cast<int>(e % Cc);
    long p = e / Cc;
    const int w = static_cast<int>(p % W), h = static_cast<int>((p / W) % H);
    const int n = static_cast<int>(p / (static_cast<long>(W) * H));
    const float g = 0.25f * dY[((static_cast<long>(n) * (H / 2) + h / 2) * (W / 2) + w / 2) * Cc + c];
    dX[e] = accumulate ? dX[e] + g : g;
}

// Y[:, :, :, 0:C1] = up2(A) (nearest), Y[:, :, :, C1:C1+C2] = Bskip
// 8 channels (16 bytes) per thread; C1 and C2 are multiples of 8 and the
// pixel count fits 32 bits
__global__ void __launch_bounds__(256) up_concat_kernel(unsigned total, unsigned H, unsigned W, unsigned G1,
                                                        unsigned G2, const bf16 *__restrict__ A,
                                                        const bf16 *__restrict__ Bk, bf16 *__restrict__ Y)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const unsigned G = G1 + G2, e = blockIdx.x * 256u + threadIdx.x;
    if (e >= total) return;
    const unsigned g = e % G, p = e / G, r = p / W, w = p % W;           // r: image and row
    const u4 *src = g < G1 ? reinterpret_cast<const u4 *>(A) +
                                 (static_cast<size_t>((r / H * (H / 2) + r % H / 2) * (W / 2) + w / 2) * G1 + g)
                           : reinterpret_cast<const u4 *>(Bk) + (static_cast<size_t>(p) * G2 + (g - G1));
    reinterpret_cast<u4 *>(Y)[e] = *src;
}

// split the gradient of up_concat: dA (low res, sum of 4) and dB (skip)
__global__ void up_concat_back_a_kernel(int Nn, int h, int w, int C1, int C2, const float *dY,
                                        float *dA)
{
    const int Ct = C1 + C2, H = 2 * h, W = 2 * w;
    const long total = static_cast<long>(Nn) * h * w * C1;
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    const int c = static_cast<int>(e % C1);
    long p = e / C1;
    const int x = static_cast<int>(p % w), y = static_cast<int>((p / w) % h);
    const int n = static_cast<int>(p / (static_cast<long>(w) * h));
    float s = 0.f;
    for (int dy = 0; dy < 2; ++dy)
        for (int dx = 0; dx < 2; ++dx)
            s += dY[((static_cast<long>(n) * H + 2 * y + dy) * W + 2 * x + dx) * Ct + c];
    dA[e] = s;
}

__global__ void up_concat_back_b_kernel(long P, int C1, int C2, const float *dY, float *dB, int accumulate)
{
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= P * C2) return;
    const long p = e / C2;
    const int c = static_cast<int>(e % C2);
    const float g = dY[p * (C1 + C2) + C1 + c];
    dB[e] = accumulate ? dB[e] + g : g;
}

__global__ void f32_to_bf16_kernel(long n, const float *a, bf16 *b)
{
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e < n) b[e] = f2bf(a[e]);
}

// mean squared error over n values; grad = 2 (y - t) / n ; loss into *loss
__global__ void mse_kernel(long n, const float *y, const float *t, float *grad, float *loss)
{
    float s = 0.f;
    for (long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; e < n;
         e += static_cast<long>(gridDim.x) * 256) {
        const float d = y[e] - t[e];
        grad[e] = 2.f * d / static_cast<float>(n);
        s += d * d;
    }
    __shared__ float red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, red[0] / static_cast<float>(n));
}

// Adam on fp32 master weights, refreshed bf16 copy
__global__ void adam_kernel(long n, float *w, bf16 *wb, const float *g, float *m, float *v,
                            float lr, float b1, float b2, float eps, float c1, float c2)
{
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= n) return;
    const float gg = g[e];
    const float mm = b1 * m[e] + (1.f - b1) * gg;
    const float vv = b2 * v[e] + (1.f - b2) * gg * gg;
    m[e] = mm;
    v[e] = vv;
    const float upd = lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    const float nw = w[e] - upd;
    w[e] = nw;
    if (wb) wb[e] = f2bf(nw);
}

__global__ void zero_kernel(long n, float *a)
{
    const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (e < n) a[e] = 0.f;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
void im2col(int n, int h, int w, int c, const bf16 *x, bf16 *col, hipStream_t st)
{
    const long t = static_cast<long>(n) * h * w * 9 * c;
    hipLaunchKernelGGL(im2col_kernel, dim3(nb(t)), dim3(256), 0, st, n, h, w, c, x, col);
}
void col2im(int n, int h, int w, int c, const float *dcol, float *dx, int acc, hipStream_t st)
{
    const long t = static_cast<long>(n) * h * w * c;
    hipLaunchKernelGGL(col2im_kernel, dim3(nb(t)), dim3(256), 0, st, n, h, w, c, dcol, dx, acc);
}
void out_fwd(long P, const bf16 *x, const bf16 *w, const float *b, float *y, hipStream_t st)
{
    hipLaunchKernelGGL(out_kernel, dim3(nb(4 * P)), dim3(256), 0, st, static_cast<unsigned>(P), x, w, b, y);
}
void relu_back(long n, const float *dy, const bf16 *y, bf16 *dz, int relu, hipStream_t st)
{
    hipLaunchKernelGGL(relu_back_kernel, dim3(nb(n)), dim3(256), 0, st, n, dy, y, dz, relu);
}
void bias_grad(long P, int c, const bf16 *dz, float *db, hipStream_t st)
{
    hipLaunchKernelGGL(bias_grad_kernel, dim3(c), dim3(256), 0, st, P, c, dz, db);
}
void pool(int n, int h, int w, int c, const bf16 *x, bf16 *y, hipStream_t st)
{
    const long t = static_cast<long>(n) * (h / 2) * (w / 2) * (c / 8);
    hipLaunchKernelGGL(pool_kernel, dim3(nb(t)), dim3(256), 0, st, static_cast<unsigned>(t), h / 2, w / 2, c / 8, x, y);
}
void pool_back(int n, int h, int w, int c, const float *dy, float *dx, int acc, hipStream_t st)
{
    const long t = static_cast<long>(n) * h * w * c;
    hipLaunchKernelGGL(pool_back_kernel, dim3(nb(t)), dim3(256), 0, st, n, h, w, c, dy, dx, acc);
}
void up_concat(int n, int h, int w, int c1, int c2, const bf16 *a, const bf16 *b, bf16 *y, hipStream_t st)
{
    const long t = static_cast<long>(n) * h * w * ((c1 + c2) / 8);
    hipLaunchKernelGGL(up_concat_kernel, dim3(nb(t)), dim3(256), 0, st, static_cast<unsigned>(t), h, w, c1 / 8, c2 / 8,
                       a, b, y);
}
void up_concat_back(int n, int h, int w, int c1, int c2, const float *dy, float *da, float *db,
                    int acc_b, hipStream_t st)
{
    const long ta = static_cast<long>(n) * (h / 2) * (w / 2) * c1;
    hipLaunchKernelGGL(up_concat_back_a_kernel, dim3(nb(ta)), dim3(256), 0, st, n, h / 2, w / 2,
                       c1, c2, dy, da);
    const long P = static_cast<long>(n) * h * w;
    hipLaunchKernelGGL(up_concat_back_b_kernel, dim3(nb(P * c2)), dim3(256), 0, st, P, c1, c2, dy,
                       db, acc_b);
}
void to_bf16(long n, const float *a, bf16 *b, hipStream_t st)
{
    hipLaunchKernelGGL(f32_to_bf16_kernel, dim3(nb(n)), dim3(256), 0, st, n, a, b);
}
void mse(long n, const float *y, const float *t, float *grad, float *loss, hipStream_t st)
{
    hipLaunchKernelGGL(mse_kernel, dim3(256), dim3(256), 0, st, n, y, t, grad, loss);
}
void adam(long n, float *w, bf16 *wb, const float *g, float *m, float *v, float lr, float b1,
          float b2, float eps, float c1, float c2, hipStream_t st)
{
    hipLaunchKernelGGL(adam_kernel, dim3(nb(n)), dim3(256), 0, st, n, w, wb, g, m, v, lr, b1, b2,
                       eps, c1, c2);
}
void zero(long n, float *a, hipStream_t st)
{
    if (n > 0) hipLaunchKernelGGL(zero_kernel, dim3(nb(n)), dim3(256), 0, st, n, a);
}
int conv3x3_cinp(int cin) { return (cin + CK - 1) / CK * CK; }
// conv3x3s_kernel's forms: tiles per wavefront and 16-byte input pieces per
// thread, which bound the width: 128 MT + 2W + 2 <= 64 NI (159).  Two tiles
// read 3 fragments for 2 MFMAs instead of 2 for 1 and stage fewer neighbours,
// but pay with fewer workgroups: not below two a CU (128 channels of 64 images of
// 8x34, 272 workgroups against 544: 14.2 against 13.0 us; 64 channels of 16x68,
// 544 against 1088: 13.7 against 15.2).
#define TBL_CONV_FORMS(X) X(2, 9) X(1, 7)
static bool conv3x3s_fits(int mt, int w, int ni) { return 128 * mt + 2 * w + 2 <= 64 * ni; }
static size_t conv3x3s_lds(int mt, int w) { return 64 * (static_cast<size_t>(9) * 32 + 128 * mt + 2 * w + 3); }
static int conv3x3s_tiles(long np, int w, int cout)
{
    return conv3x3s_fits(2, w, 9) && (np + 255) / 256 * (cout / 32) >= 512 ? 2 : 1;
}
void pack_conv3x3(int cin, int cout, const bf16 *w, bf16 *wp, hipStream_t st)
{
    const int cinp = conv3x3_cinp(cin);
    hipLaunchKernelGGL(pack_conv3x3_kernel, dim3(nb(9L * cout * cinp)), dim3(256), 0, st, cin, cinp,
                       cout, w, wp);
}
void conv3x3(int n, int h, int w, int cin, int cout, const bf16 *x, const bf16 *wp,
             const float *bias, bf16 *y, int relu, hipStream_t st)
{
    const int cinp = conv3x3_cinp(cin);
    const long np = static_cast<long>(n) * h * w;
    // the staged form: whole chunks of channels or the first layer's four, 32-bit
    // pixel and byte counts of a tile, and a reach that its pieces hold
    if (cout % 32 == 0 && (cin % CK == 0 || cin == 4) && np < (1L << 31) - 512 &&
        conv3x3s_fits(1, w, 7) && static_cast<long>(cout) * cinp * 18 < (1L << 31)) {
        static const bool staged_ok = [] {
            bool ok = true;
#define X(MT, NI)                                                                              \
    for (const void *f : {reinterpret_cast<const void *>(&conv3x3s_kernel<MT, NI, false>),     \
                          reinterpret_cast<const void *>(&conv3x3s_kernel<MT, NI, true>)})     \
        ok = ok && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
            TBL_CONV_FORMS(X)
#undef X
            return ok;
        }();
        const int mt = conv3x3s_tiles(np, w, cout);
#define X(MT, NI)                                                                              \
    if (staged_ok && mt == MT) {                                                               \
        const dim3 grid(static_cast<unsigned>((np + 128 * MT - 1) / (128 * MT)), cout / 32);   \
        if (cin == 4)                                                                          \
            hipLaunchKernelGGL((conv3x3s_kernel<MT, NI, true>), grid, dim3(256),               \
                               conv3x3s_lds(MT, w), st, static_cast<int>(np), h, w, cin, cinp, \
                               cout, x, wp, bias, y, relu);                                    \
        else                                                                                   \
            hipLaunchKernelGGL((conv3x3s_kernel<MT, NI, false>), grid, dim3(256),              \
                               conv3x3s_lds(MT, w), st, static_cast<int>(np), h, w, cin, cinp, \
                               cout, x, wp, bias, y, relu);                                    \
        return;                                                                                \
    }
        TBL_CONV_FORMS(X)
#undef X
    }
    if (cout % 64 == 0) {
        dim3 grid(static_cast<unsigned>((np + 63) / 64), cout / 64);
        hipLaunchKernelGGL(conv3x3_kernel<64>, grid, dim3(256), 0, st, np, h, w, cin, cinp, cout, x,
                           wp, bias, y, relu);
    } else {
        dim3 grid(static_cast<unsigned>((np + 127) / 128), cout / 32);
        hipLaunchKernelGGL(conv3x3_kernel<32>, grid, dim3(256), 0, st, np, h, w, cin, cinp, cout, x,
                           wp, bias, y, relu);
    }
}


// ---- backward launchers ------------------------------------------------------
constexpr size_t kBwdLds = 160 * 1024;
// conv3x3_dx_kernel's forms: pixel tiles a wavefront, tiles of 32 input channels a
// workgroup, output channels
#define TBL_DX_SHAPES(X) X(2, 1, 32) X(2, 1, 64) X(1, 2, 64) X(1, 2, 128) X(1, 2, 256)
static int dx_nt(int cin, int cout) { return cin % 64 == 0 && cout != 32 ? 2 : 1; }
static size_t dx_lds(int px, int w, int ct, int cout)
{
    return static_cast<size_t>(px + 2 * w + 2 + ct) * (cout + 8) * sizeof(bf16);
}
// rows per group of conv3x3_dw_kernel: about 256 / NC pixels, which keeps two
// workgroups' tiles on a CU
static int dw_rows(int w, int nc) { return std::max(1, ((nc == 4 ? 128 : nc == 2 ? 192 : 256) + w / 2) / w); }
static size_t dw_lds(int w, int nc)
{
    const int nr = dw_rows(w, nc), np = (nr * w + 31) / 32 * 32;
    return dw_x_bytes(nr, w) + static_cast<size_t>(nc) * np * kWgRow * sizeof(bf16) +
           3 * np * sizeof(uint16_t);
}
static int dw_chunks(int cout) { return cout % 128 == 0 ? 4 : cout % 64 == 0 ? 2 : 1; }
// the direct backward kernels take a layer whose tiles fit (widths up to about
// 500) and whose staged rows fit 16-bit offsets
bool conv3x3_back_fits(int w, int cin, int cout)
{
    const int nc = dw_chunks(cout);
    const int nt = dx_nt(cin, cout);
    bool form = false;
#define X(MT, NT, CO) form = form || (nt == NT && cout == CO);
    TBL_DX_SHAPES(X)
#undef X
    return form && cin % 4 == 0 && dw_lds(w, nc) <= kBwdLds &&
           dx_lds(128 * (3 - nt), w, 32 * nt, cout) <= kBwdLds &&
           static_cast<long>(dw_rows(w, nc) + 3) * (w + 2) * (kWgRow / 4) < 65536;
}
// slices of the weight gradient's workspace: enough workgroups for the chip on
// the wide levels, fewer where a slice is large (its write and read grow with it)
int conv3x3_dw_slices(int n, int h, int w, int cin, int cout)
{
    const int nc = dw_chunks(cout), rows = n * h, nr = dw_rows(w, nc);
    const int blocks = (cin + 31) / 32 * (cout / (32 * nc));
    return std::max(1, std::min((rows + nr - 1) / nr, (nc == 1 ? 512 : 256) / blocks));
}
int relu_back_slices(long P) { return static_cast<int>(std::max(1L, std::min(512L, P / 64))); }

void conv3x3_dw(int n, int h, int w, int cin, int cout, const bf16 *x, const bf16 *dz, float *ws,
                hipStream_t st)
{
    const int nc = dw_chunks(cout), nr = dw_rows(w, nc), ks = (nr * w + 31) / 32;
    const dim3 grid(conv3x3_dw_slices(n, h, w, cin, cout), (cin + 31) / 32, cout / (32 * nc));
    const size_t lds = dw_lds(w, nc);
    if (nc == 4)
        hipLaunchKernelGGL(conv3x3_dw_kernel<4>, grid, dim3(256), lds, st, n * h, h, w, nr, ks, cin, cout, x, dz, ws);
    else if (nc == 2)
        hipLaunchKernelGGL(conv3x3_dw_kernel<2>, grid, dim3(256), lds, st, n * h, h, w, nr, ks, cin, cout, x, dz, ws);
    else
        hipLaunchKernelGGL(conv3x3_dw_kernel<1>, grid, dim3(256), lds, st, n * h, h, w, nr, ks, cin, cout, x, dz, ws);
}

void conv3x3_dx(int n, int h, int w, int cin, int cout, const bf16 *dz, const bf16 *wb, float *dx,
                hipStream_t st)
{
    const long np = static_cast<long>(n) * h * w;
    const int nt = dx_nt(cin, cout), px = 128 * (3 - nt);
    const dim3 grid(static_cast<unsigned>((np + px - 1) / px), (cin + 32 * nt - 1) / (32 * nt));
#define X(MT, NT, CO)                                                                            \
    if (nt == NT && cout == CO) {                                                                \
        hipLaunchKernelGGL((conv3x3_dx_kernel<MT, NT, CO>), grid, dim3(256),                     \
                           dx_lds(px, w, 32 * NT, CO), st, np, h, w, cin, dz, wb, dx);           \
        return;                                                                                  \
    }
    TBL_DX_SHAPES(X)
#undef X
}
void wgrad_reduce(int n, int slices, const float *ws, float *g, int cout, int bslices, const float *bs,
                  float *gb, hipStream_t st)
{
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((n + cout + 63) / 64), dim3(256), 0, st, n, slices, ws, g, cout,
                       bslices, bs, gb);
}
void relu_back_bias(long P, int c, const float *dy, const bf16 *y, bf16 *dz, float *bs, hipStream_t st)
{
    const int s = relu_back_slices(P);
    hipLaunchKernelGGL(relu_back_bias_kernel, dim3(s), dim3(256), 0, st, P, c, (P + s - 1) / s, dy, y, dz, bs);
}
void out_back(long P, const float *dy, const bf16 *x, const bf16 *w, float *dx, float *ws, float *bs,
              hipStream_t st)
{
    const int s = relu_back_slices(P);
    hipLaunchKernelGGL(out_back_kernel, dim3(s), dim3(256), 0, st, P, (P + s - 1) / s, dy, x, w, dx, ws, bs);
}
int nn_kernel_attributes()
{
    hipError_t e = hipSuccess;
    auto allow = [&](const void *f) {
        const hipError_t r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kBwdLds);
        if (r != hipSuccess) e = r;
    };
#define X(MT, NT, CO) allow(reinterpret_cast<const void *>(&conv3x3_dx_kernel<MT, NT, CO>));
    TBL_DX_SHAPES(X)
#undef X
    allow(reinterpret_cast<const void *>(&conv3x3_dw_kernel<1>));
    allow(reinterpret_cast<const void *>(&conv3x3_dw_kernel<2>));
    allow(reinterpret_cast<const void *>(&conv3x3_dw_kernel<4>));
    return e == hipSuccess ? TBL_OK : TBL_ERR_HIP;
}

}  // namespace nn
}  // namespace tbl
