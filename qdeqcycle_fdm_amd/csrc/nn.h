// nn.h -- host launchers of the learned-guess network kernels (nn.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace qdeq {
namespace nn {

typedef __bf16 bf16;

enum { GEMM_CFG_WIDE = 0, GEMM_CFG_SKINNY = 1 };
enum { EPI_PLAIN = 0, EPI_RELU = 1 };

// What a GEMM does with its result C [M x N]:
//   OUT_F32   outF = C
//   OUT_RELU  out, outT = bf16(max(C, 0)) and its transpose
//   OUT_MASK  C where mask > 0, else 0: into out and outT, or outF (FP32)
//   OUT_MSE   C is the network's output: the mean squared error against rows
//             idx[b] (b without idx) of target, b < B, columns < nout; out and
//             outT = the gradient of C, partial = a sum per block of 128 x 128
//   OUT_ADAM  C is the gradient of the weights outF [M x N]: Adam with the
//             moments m and v; out, outT = the BF16 copies of the new weights
enum { OUT_F32 = 0, OUT_RELU = 1, OUT_MASK = 2, OUT_MSE = 3, OUT_ADAM = 4 };
enum { kWideBlocks = 128, kMaxWaveSplits = 8 };

struct AdamCoef {
  float lr, b1, b2, eps, c1, c2;
};

struct GemmOut {
  bf16 *out, *outT;
  float *outF;
  const bf16 *mask;
  const float *target;
  const int *idx;
  int B, nout;
  double *partial;
  float *m, *v;
  AdamCoef adam;
};

// C[M x N] = A[M x K] * B[N x K]^T, BF16 operands with row pitches lda, ldb
// (multiples of 8), FP32 accumulation; M, N multiples of 128, K of 32.  K is
// split into chunks whose FP32 sums are added in order when fewer than 512
// blocks of 128 x 128 would run (splitbuf holds them where the chunks are too
// many for one block).  Returns -1 on shapes the kernels do not cover
// (nothing is launched then).
bool gemm_shape_ok(int cfg, int M, int N, int K, int lda, int ldb);
int gemm(hipStream_t st, int out, const bf16 *A, int lda, const bf16 *B, int ldb, int M, int N,
         int K, float *splitbuf, size_t splitbuf_floats, const GemmOut &o);

// C (FP32, pitch N) for few rows: M % 16 == 0, N % 128 == 0, K % 32 == 0.
int gemm_skinny(hipStream_t st, const bf16 *A, int lda, const bf16 *B, int ldb,
                float *C, int M, int N, int K, float *splitbuf,
                size_t splitbuf_floats, int min_blocks);

// out / outT (BF16, optional) = op(Z) and its transpose.  Z is M x N row-major.
void epilogue(hipStream_t st, const float *Z, int M, int N, int mode, bf16 *out,
              bf16 *outT);

// Encoder Conv1d(1 -> C, width T, stride S) + ReLU on rows idx[b] (b without
// idx) of X [. x nk] (FP32), b < B; rows B..M-1 are zero: H0 [M x P0*C] and
// H0T [P0*C x M] (optional), feature p*C + c.
void conv_forward(hipStream_t st, const float *X, const int *idx, int B, int M, int nk,
                  const float *Wc, int C, int T, int S, int P0, bf16 *H0, bf16 *H0T);
// Its weights' gradient into gWc, or with w the Adam update of w, m, v; and
// *loss = scale * the sum of partial[0..npart).
void conv_backward(hipStream_t st, const float *X, const int *idx, int B, int nk,
                   const float *dZ0, int C, int T, int S, int P0, float *gWc, float *w,
                   float *m, float *v, const AdamCoef &k, const double *partial, int npart,
                   double scale, double *loss);

}  // namespace nn
}  // namespace qdeq
