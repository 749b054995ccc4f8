// BF16 U-Net of the learned initial guess: kernel launchers and the network
// object behind the tbl_net handle.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace tbl {
namespace nn {

typedef uint16_t bf16;   // bfloat16 bit pattern

void gemm(int M, int N, int K, const bf16 *A, long sam, long sak, const bf16 *B, long sbk,
          long sbn, float *C, long ldc, float alpha, float beta, hipStream_t st, int splitk = 1);
void im2col(int n, int h, int w, int c, const bf16 *x, bf16 *col, hipStream_t st);
void col2im(int n, int h, int w, int c, const float *dcol, float *dx, int acc, hipStream_t st);
void out_fwd(long P, const bf16 *x, const bf16 *w, const float *b, float *y, hipStream_t st);
void relu_back(long n, const float *dy, const bf16 *y, bf16 *dz, int relu, hipStream_t st);
void bias_grad(long P, int c, const bf16 *dz, float *db, hipStream_t st);
void pool(int n, int h, int w, int c, const bf16 *x, bf16 *y, hipStream_t st);
void pool_back(int n, int h, int w, int c, const float *dy, float *dx, int acc, hipStream_t st);
void up_concat(int n, int h, int w, int c1, int c2, const bf16 *a, const bf16 *b, bf16 *y,
               hipStream_t st);
void up_concat_back(int n, int h, int w, int c1, int c2, const float *dy, float *da, float *db,
                    int acc_b, hipStream_t st);
void to_bf16(long n, const float *a, bf16 *b, hipStream_t st);
void mse(long n, const float *y, const float *t, float *grad, float *loss, hipStream_t st);
void adam(long n, float *w, bf16 *wb, const float *g, float *m, float *v, float lr, float b1,
          float b2, float eps, float c1, float c2, hipStream_t st);
void zero(long n, float *a, hipStream_t st);
// direct 3x3 convolution + bias (+ ReLU) -> bf16 NHWC; weights packed by
// pack_conv3x3 into [tap][cout][cin rounded up to 32]; cout a multiple of 32
int conv3x3_cinp(int cin);
void pack_conv3x3(int cin, int cout, const bf16 *w, bf16 *wp, hipStream_t st);
void conv3x3(int n, int h, int w, int cin, int cout, const bf16 *x, const bf16 *wp,
             const float *bias, bf16 *y, int relu, hipStream_t st);

// direct backward of a 3x3 convolution (where conv3x3_back_fits): dz = dy * (y >
// 0) with bias partials bs [relu_back_slices][c], weight-gradient partials ws
// [conv3x3_dw_slices][9 cin cout], their sums, and the input's gradient from
// the unpacked weights [tap][cin][cout]
bool conv3x3_back_fits(int w, int cin, int cout);
int conv3x3_dw_slices(int n, int h, int w, int cin, int cout);
int relu_back_slices(long P);
void relu_back_bias(long P, int c, const float *dy, const bf16 *y, bf16 *dz, float *bs, hipStream_t st);
void conv3x3_dw(int n, int h, int w, int cin, int cout, const bf16 *x, const bf16 *dz, float *ws,
                hipStream_t st);
void wgrad_reduce(int n, int slices, const float *ws, float *g, int cout, int bslices, const float *bs,
                  float *gb, hipStream_t st);
void conv3x3_dx(int n, int h, int w, int cin, int cout, const bf16 *dz, const bf16 *wb, float *dx,
                hipStream_t st);
// the 1x1 output layer (32 channels in, 2 out): dx, and partials ws [][64], bs [][2]
void out_back(long P, const float *dy, const bf16 *x, const bf16 *w, float *dx, float *ws, float *bs,
              hipStream_t st);
int nn_kernel_attributes();

}  // namespace nn
}  // namespace tbl
