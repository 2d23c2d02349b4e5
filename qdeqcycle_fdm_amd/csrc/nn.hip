// nn.hip -- kernels of the learned initial guess network: BF16 MFMA GEMMs
// with FP32 accumulation (gfx950 v_mfma_f32_16x16x32_bf16) whose last step is
// the activation, the mask, the MSE loss or the Adam update, and the 1D
// convolution encoder.  No reference counterpart: the reference starts every
// elliptic solve from the previous solution (odeSolver.cpp:652-720); this
// network predicts a better start.
//
// GEMM convention: C[M x N] = A[M x K] * B[N x K]^T with A and B row-major
// in their K dimension (both operands K-contiguous).  Every product of the
// forward and backward pass is written in this form by keeping transposed
// BF16 copies of the weights, activations and gradients; the kernel that
// computes a matrix writes both copies.
//
// A training step is bound by launches and by passes over memory, not by the
// matrix cores: at 513 fault nodes (batch 160 padded to 256 rows, 9.7 M
// parameters) its products take 11 GFLOP, 10 us of the card, and Adam's seven
// words per parameter 270 MB, 55 us.  With the last steps in kernels of their
// own (split sums, activation and transposes, loss, Adam, BF16 copies,
// minibatch gather) a step took 41 launches and 430 us; it takes 15 launches
// and 213 us: 58 the last layer's gradient with its Adam, 24 the output with
// the loss, 30 the gradient through the last layer, 17 the encoder's gradient.

#include "nn.h"

#include <algorithm>

namespace qdeq {
namespace nn {

typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---- what a GEMM does with its result ----

// Adam (bias-corrected), FP32 master weights.
__device__ inline void adam_step(const AdamCoef &k, float g, float &w, float &m, float &v) {
  const float mi = k.b1 * m + (1.f - k.b1) * g;
  const float vi = k.b2 * v + (1.f - k.b2) * g * g;
  m = mi;
  v = vi;
  w = w - k.lr * (mi / k.c1) / (sqrtf(vi / k.c2) + k.eps);
}

// What the last step reads for four elements of a row, (row, col..col+3), col
// a multiple of 4.
struct Fetched {
  f32x4 a, m, v;  // target or weights, moments
  bf16x4 mask;
};

template <int OUT>
__device__ inline Fetched fetch4(const GemmOut &o, int N, int row, int col, int src) {
  const long long i = (long long)row * N + col;
  Fetched f;
  if (OUT == OUT_MASK) f.mask = *reinterpret_cast<const bf16x4 *>(o.mask + i);
  if (OUT == OUT_MSE) f.a = *reinterpret_cast<const f32x4 *>(o.target + (long long)src * N + col);
  if (OUT == OUT_ADAM) {
    f.a = *reinterpret_cast<const f32x4 *>(o.outF + i);
    f.m = *reinterpret_cast<const f32x4 *>(o.m + i);
    f.v = *reinterpret_cast<const f32x4 *>(o.v + i);
  }
  return f;
}

// Row of the loss's target for row b of the batch (any row for the padding).
template <int OUT>
__device__ inline int target_row(const GemmOut &o, int b) {
  if (OUT != OUT_MSE) return 0;
  b = min(b, o.B - 1);
  return o.idx ? o.idx[b] : b;
}

// The last step on four elements c of a row.  Returns the values that the BF16
// copies hold.
template <int OUT>
__device__ inline f32x4 finish4(const GemmOut &o, int N, int row, int col, f32x4 c,
                                const Fetched &f, double &loss) {
  const long long i = (long long)row * N + col;
  if (OUT == OUT_F32) {
    *reinterpret_cast<f32x4 *>(o.outF + i) = c;
  } else if (OUT == OUT_RELU) {
#pragma unroll
    for (int e = 0; e < 4; e++) c[e] = c[e] > 0.f ? c[e] : 0.f;
  } else if (OUT == OUT_MASK) {
#pragma unroll
    for (int e = 0; e < 4; e++) c[e] = (float)f.mask[e] > 0.f ? c[e] : 0.f;
    if (o.outF) *reinterpret_cast<f32x4 *>(o.outF + i) = c;
  } else if (OUT == OUT_MSE) {
    // rows >= B and the padding columns >= nout: gradient zero, no loss
    const float scale = 2.0f / ((float)o.B * (float)o.nout);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float g = 0.f;
      if (row < o.B && col + e < o.nout) {
        const float d = c[e] - f.a[e];
        loss += (double)d * (double)d;
        g = scale * d;
      }
      c[e] = g;
    }
  } else if (OUT == OUT_ADAM) {
    f32x4 w = f.a, m = f.m, v = f.v;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float we = w[e], me = m[e], ve = v[e];
      adam_step(o.adam, c[e], we, me, ve);
      w[e] = we;
      m[e] = me;
      v[e] = ve;
    }
    *reinterpret_cast<f32x4 *>(o.outF + i) = w;
    *reinterpret_cast<f32x4 *>(o.m + i) = m;
    *reinterpret_cast<f32x4 *>(o.v + i) = v;
    c = w;
  }
  return c;
}

__device__ inline bf16x4 to_bf16x4(f32x4 c) {
  return bf16x4{(bf16)c[0], (bf16)c[1], (bf16)c[2], (bf16)c[3]};
}

// ---- GEMM, wide ----
// Block = 2 x 2 wavefronts; each computes 4 x 4 tiles of 16x16 with the
// 16x16x32 MFMA.  K is consumed 32 at a time through a double-buffered LDS
// stage (rows padded to 40 elements = 80 bytes).  Operand lanes: lane l feeds
// row/column (l & 15) and the k-group (l >> 4) of eight consecutive k values,
// the same k-group for both operands.  The B fragment is the MFMA's first
// operand, so result element r of lane l is row (l & 15), column
// 4*(l >> 4) + r of the tile: four neighbours of a row, loaded and stored as
// 16 bytes by the last step.
// blockIdx.z selects a K chunk [z*kchunk, (z+1)*kchunk) and the FP32 output
// slice o.outF + z*split_stride (partial sums, added by k_split_finish).  With
// FOLD a block computes all `folds` chunks one after the other and adds their
// sums in order: the same result without the partial sums in memory.  Few
// blocks run per CU, so the loads of two k-steps are in flight and registers
// are held to two blocks a CU (one took 42 us for the output and loss, 24 now).
template <int WM, int WN, int TM, int TN, bool FOLD, int OUT>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_gemm_nt(
    const bf16 *__restrict__ A, int lda, const bf16 *__restrict__ B, int ldb,
    int M, int N, int kchunk, int folds, long long split_stride, GemmOut o) {
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16, BK = 32;
  constexpr int NT = 64 * WM * WN, LDK = BK + 8;
  constexpr int ACH = BM * BK / 8, BCH = BN * BK / 8;
  constexpr int AIT = (ACH + NT - 1) / NT, BIT = (BCH + NT - 1) / NT;
  constexpr int TP = 16 * TM + 8;  // pitch of a wavefront's transposed tile
  constexpr bool COPIES = OUT != OUT_F32;
  constexpr int STAGE = 2 * (BM + BN) * LDK;
  static_assert(!COPIES || WM * WN * 16 * TN * TP <= STAGE, "transposed tiles reuse the stage");
  __shared__ __attribute__((aligned(16))) bf16 sm[STAGE];
  bf16 *const As = sm, *const Bs = sm + 2 * BM * LDK;

  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int kbeg = blockIdx.z * kchunk, kend = kbeg + kchunk * (FOLD ? folds : 1);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;

  f32x4 acc[TM][TN], sum[FOLD ? TM : 1][FOLD ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Stage {
    bf16x8 a[AIT], b[BIT];
  } r0, r1;
  auto gload = [&](int k, Stage &r) {
#pragma unroll
    for (int i = 0; i < AIT; i++) {
      const int ch = tid + i * NT;
      if (ACH % NT == 0 || ch < ACH) {
        const int row = ch >> 2, kk = (ch & 3) * 8;
        r.a[i] = *reinterpret_cast<const bf16x8 *>(A + (long long)(m0 + row) * lda + k + kk);
      }
    }
#pragma unroll
    for (int i = 0; i < BIT; i++) {
      const int ch = tid + i * NT;
      if (BCH % NT == 0 || ch < BCH) {
        const int row = ch >> 2, kk = (ch & 3) * 8;
        r.b[i] = *reinterpret_cast<const bf16x8 *>(B + (long long)(n0 + row) * ldb + k + kk);
      }
    }
  };
  auto sstore = [&](int buf, const Stage &r) {
#pragma unroll
    for (int i = 0; i < AIT; i++) {
      const int ch = tid + i * NT;
      if (ACH % NT == 0 || ch < ACH) {
        const int row = ch >> 2, kk = (ch & 3) * 8;
        *reinterpret_cast<bf16x8 *>(As + (buf * BM + row) * LDK + kk) = r.a[i];
      }
    }
#pragma unroll
    for (int i = 0; i < BIT; i++) {
      const int ch = tid + i * NT;
      if (BCH % NT == 0 || ch < BCH) {
        const int row = ch >> 2, kk = (ch & 3) * 8;
        *reinterpret_cast<bf16x8 *>(Bs + (buf * BN + row) * LDK + kk) = r.b[i];
      }
    }
  };

  const int ar = wm * TM * 16 + (lane & 15), br = wn * TN * 16 + (lane & 15);
  const int kg = (lane >> 4) * 8;
  int kfold = kbeg + kchunk;
  // k-step at k from LDS stage buf; `next` holds the loads of the step after it,
  // `after` receives those of the second one
  auto step = [&](int k, int buf, const Stage &next, Stage &after) {
    if (k + 2 * BK < kend) gload(k + 2 * BK, after);
    bf16x8 a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
      a[i] = *reinterpret_cast<const bf16x8 *>(As + (buf * BM + ar + i * 16) * LDK + kg);
#pragma unroll
    for (int j = 0; j < TN; j++)
      b[j] = *reinterpret_cast<const bf16x8 *>(Bs + (buf * BN + br + j * 16) * LDK + kg);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
    if (FOLD && k + BK == kfold) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          sum[i][j] = kfold == kbeg + kchunk ? acc[i][j] : sum[i][j] + acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      kfold += kchunk;
    }
    if (k + BK < kend) sstore(buf ^ 1, next);
    __syncthreads();
  };
  gload(kbeg, r0);
  if (kbeg + BK < kend) gload(kbeg + BK, r1);
  sstore(0, r0);
  __syncthreads();
  for (int k = kbeg; k < kend; k += 2 * BK) {
    step(k, 0, r1, r0);
    if (k + BK < kend) step(k + BK, 1, r0, r1);
  }
  const int rbase = m0 + wm * TM * 16, cbase = n0 + wn * TN * 16;
  bf16 *const tile = sm + wave * 16 * TN * TP;
  double loss = 0.0;
  if (OUT == OUT_F32) o.outF += (long long)blockIdx.z * split_stride;
  // a row of tiles' inputs are fetched before its first store
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int r = i * 16 + (lane & 15), src = target_row<OUT>(o, rbase + r);
    Fetched f[TN];
#pragma unroll
    for (int j = 0; j < TN; j++)
      f[j] = fetch4<OUT>(o, N, rbase + r, cbase + j * 16 + 4 * (lane >> 4), src);
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int c = j * 16 + 4 * (lane >> 4);
      const f32x4 v =
          finish4<OUT>(o, N, rbase + r, cbase + c, FOLD ? sum[i][j] : acc[i][j], f[j], loss);
      if (COPIES && o.out) {
        const bf16x4 h = to_bf16x4(v);
        *reinterpret_cast<bf16x4 *>(o.out + (long long)(rbase + r) * N + cbase + c) = h;
#pragma unroll
        for (int e = 0; e < 4; e++) tile[(c + e) * TP + r] = h[e];
      }
    }
  }
  if (!COPIES || !o.outT) return;
  // the transposed copy, 16 bytes of a wavefront's own tile per lane
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int q = lane; q < 16 * TN * (2 * TM); q += 64) {
    const int c = q / (2 * TM), r = (q % (2 * TM)) * 8;
    *reinterpret_cast<bf16x8 *>(o.outT + (long long)(cbase + c) * M + rbase + r) =
        *reinterpret_cast<const bf16x8 *>(tile + c * TP + r);
  }
  if (OUT == OUT_MSE) {
    __shared__ double red[WM * WN];
    for (int d = 32; d > 0; d >>= 1) loss += __shfl_down(loss, d);
    if (lane == 0) red[wave] = loss;
    __syncthreads();
    if (tid == 0) {
      double s = red[0];
      for (int w = 1; w < WM * WN; w++) s += red[w];
      o.partial[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = s;
    }
  }
}

// ---- GEMM, K split over the wavefronts of a block ----
// For products of fewer than kWideBlocks wide blocks (hidden layers: 256 x 512,
// K = 512), where a wide block's chain of loads leaves most of the card idle
// and the split sums cost two more launches.  Block = one 32 x 32 tile;
// wavefront z computes K chunk z with its fragments straight from memory (all
// loads of 128 k at once), the partial sums are added through LDS in chunk
// order.  256 x 512 x 512 with its activation and transposed copy: 12.5 us as
// a wide split product, its sum and its epilogue, 4.8 us here.
constexpr int kPP = 36;  // row pitch of a partial tile: no bank conflicts

template <int OUT>
__global__ __launch_bounds__(64 * kMaxWaveSplits) void k_gemm_waves(
    const bf16 *__restrict__ A, int lda, const bf16 *__restrict__ B, int ldb,
    int M, int N, int kchunk, GemmOut o) {
  extern __shared__ __attribute__((aligned(16))) float part[];
  __shared__ __attribute__((aligned(16))) bf16 tile[32 * kPP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int waves = blockDim.x >> 6;
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  const long long k0 = (long long)wave * kchunk + (lane >> 4) * 8;
  const bf16 *a0 = A + (long long)(m0 + (lane & 15)) * lda + k0, *a1 = a0 + 16LL * lda;
  const bf16 *b0 = B + (long long)(n0 + (lane & 15)) * ldb + k0, *b1 = b0 + 16LL * ldb;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](bf16x8 x0, bf16x8 x1, bf16x8 y0, bf16x8 y1) {
    acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y0, x0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y1, x0, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y0, x1, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y1, x1, acc[1][1], 0, 0, 0);
  };
  auto frag = [](const bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); };
  int k = 0;
  for (; k + 128 <= kchunk; k += 128) {
    bf16x8 x0[4], x1[4], y0[4], y1[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      x0[u] = frag(a0 + k + 32 * u);
      x1[u] = frag(a1 + k + 32 * u);
      y0[u] = frag(b0 + k + 32 * u);
      y1[u] = frag(b1 + k + 32 * u);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) mul(x0[u], x1[u], y0[u], y1[u]);
  }
  for (; k < kchunk; k += 32) mul(frag(a0 + k), frag(a1 + k), frag(b0 + k), frag(b1 + k));
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
      *reinterpret_cast<f32x4 *>(part + (wave * 32 + i * 16 + (lane & 15)) * kPP + j * 16 +
                                 4 * (lane >> 4)) = acc[i][j];
  __syncthreads();
  double loss = 0.0;
  for (int q = tid; q < 256; q += blockDim.x) {
    const int r = q >> 3, c = (q & 7) * 4;
    f32x4 s = *reinterpret_cast<const f32x4 *>(part + r * kPP + c);
    for (int z = 1; z < waves; z++)
      s = s + *reinterpret_cast<const f32x4 *>(part + (z * 32 + r) * kPP + c);
    const Fetched f = fetch4<OUT>(o, N, m0 + r, n0 + c, 0);
    const f32x4 v = finish4<OUT>(o, N, m0 + r, n0 + c, s, f, loss);
    if (o.out) {
      const bf16x4 h = to_bf16x4(v);
      *reinterpret_cast<bf16x4 *>(o.out + (long long)(m0 + r) * N + n0 + c) = h;
#pragma unroll
      for (int e = 0; e < 4; e++) tile[(c + e) * kPP + r] = h[e];
    }
  }
  if (!o.outT) return;
  __syncthreads();
  for (int q = tid; q < 256; q += blockDim.x) {
    const int c = q >> 3, r = (q & 7) * 4;
    *reinterpret_cast<bf16x4 *>(o.outT + (long long)(n0 + c) * M + m0 + r) =
        *reinterpret_cast<const bf16x4 *>(tile + c * kPP + r);
  }
}

// Sum of the K chunks' partial results (M x N each) in chunk order, and the
// last step.  Block = 32 x 32 elements, 16 partial sums in flight per thread.
template <int OUT>
__global__ __launch_bounds__(256) void k_split_finish(const float *__restrict__ part, int splits,
                                                      int M, int N, GemmOut o) {
  __shared__ __attribute__((aligned(16))) bf16 tile[32 * kPP];
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  const int hi = threadIdx.x >> 3, lo = (threadIdx.x & 7) * 4;
  const long long mn = (long long)M * N;
  const float *p = part + (long long)(m0 + hi) * N + n0 + lo;
  f32x4 s = *reinterpret_cast<const f32x4 *>(p);
  int z = 1;
  for (; z + 16 <= splits; z += 16) {
    f32x4 t[16];
#pragma unroll
    for (int u = 0; u < 16; u++) t[u] = *reinterpret_cast<const f32x4 *>(p + (z + u) * mn);
#pragma unroll
    for (int u = 0; u < 16; u++) s = s + t[u];
  }
#pragma unroll 4
  for (; z < splits; z++) s = s + *reinterpret_cast<const f32x4 *>(p + z * mn);
  double loss = 0.0;
  const Fetched f = fetch4<OUT>(o, N, m0 + hi, n0 + lo, 0);
  const f32x4 v = finish4<OUT>(o, N, m0 + hi, n0 + lo, s, f, loss);
  if (o.out) {
    const bf16x4 h = to_bf16x4(v);
    *reinterpret_cast<bf16x4 *>(o.out + (long long)(m0 + hi) * N + n0 + lo) = h;
#pragma unroll
    for (int e = 0; e < 4; e++) tile[(lo + e) * kPP + hi] = h[e];
  }
  if (!o.outT) return;
  __syncthreads();
  *reinterpret_cast<bf16x4 *>(o.outT + (long long)(n0 + hi) * M + m0 + lo) =
      *reinterpret_cast<const bf16x4 *>(tile + hi * kPP + lo);
}

// Tile configurations: "wide" for training (128 x 128 per block), "skinny"
// for the 16-row inference products (16 x 128 per block).
#define GEMM_WIDE 2, 2, 4, 4
#define GEMM_SKINNY 1, 4, 1, 2

bool gemm_shape_ok(int cfg, int M, int N, int K, int lda, int ldb) {
  const int BM = cfg == GEMM_CFG_WIDE ? 128 : 16;
  const int BN = 128;
  return M > 0 && N > 0 && K > 0 && M % BM == 0 && N % BN == 0 && K % 32 == 0 &&
         lda % 8 == 0 && ldb % 8 == 0 && lda >= K && ldb >= K;
}

// Smallest split of K into equal whole chunks that gives min_blocks blocks (at
// most 64 chunks of at least 4 k-steps; FP32 partials must fit).
static int gemm_splits(int blocks, long long mn, int K, size_t splitbuf_floats, int min_blocks) {
  const int nk32 = K / 32;
  int splits = 1;
  for (int s = 2; s <= 64 && blocks * splits < min_blocks; s++) {
    if (nk32 % s || nk32 / s < 4) continue;
    if ((size_t)s * (size_t)mn > splitbuf_floats) break;
    splits = s;
  }
  return splits;
}

template <int OUT>
static void gemm_out(hipStream_t st, const bf16 *A, int lda, const bf16 *B, int ldb, int M,
                     int N, int K, float *splitbuf, size_t splitbuf_floats, const GemmOut &o) {
  const int gm = M / 128, gn = N / 128;
  const int splits = gemm_splits(gm * gn, (long long)M * N, K, splitbuf_floats, 512);
  const int kchunk = K / splits;
  const dim3 grid(gn, gm), tiles(N / 32, M / 32);
  // From 128 wide blocks (half the card's CUs) on, a quarter of the operand
  // traffic is worth more than the other CUs: the last layer's 132 x 4 blocks of
  // 256 k take 15 us wide and would read four times the operands as 32 x 32 tiles.
  if (OUT == OUT_MSE || gm * gn >= kWideBlocks) {
    if (splits > 1)
      hipLaunchKernelGGL((k_gemm_nt<GEMM_WIDE, true, OUT>), grid, dim3(256), 0, st, A, lda, B,
                         ldb, M, N, kchunk, splits, 0LL, o);
    else
      hipLaunchKernelGGL((k_gemm_nt<GEMM_WIDE, false, OUT>), grid, dim3(256), 0, st, A, lda, B,
                         ldb, M, N, kchunk, 1, 0LL, o);
    return;
  }
  if constexpr (OUT == OUT_MSE) {
    return;  // always wide: its loss is summed per wide block
  } else if (splits <= kMaxWaveSplits) {
    hipLaunchKernelGGL((k_gemm_waves<OUT>), tiles, dim3(64 * splits),
                       (size_t)splits * 32 * kPP * sizeof(float), st, A, lda, B, ldb, M, N,
                       kchunk, o);
  } else {
    GemmOut p{};
    p.outF = splitbuf;
    hipLaunchKernelGGL((k_gemm_nt<GEMM_WIDE, false, OUT_F32>), dim3(gn, gm, splits), dim3(256),
                       0, st, A, lda, B, ldb, M, N, kchunk, 1, (long long)M * N, p);
    hipLaunchKernelGGL((k_split_finish<OUT>), tiles, dim3(256), 0, st, splitbuf, splits, M, N,
                       o);
  }
}

int gemm(hipStream_t st, int out, const bf16 *A, int lda, const bf16 *B, int ldb, int M, int N,
         int K, float *splitbuf, size_t splitbuf_floats, const GemmOut &o) {
  if (!gemm_shape_ok(GEMM_CFG_WIDE, M, N, K, lda, ldb)) return -1;
  switch (out) {
    case OUT_F32: gemm_out<OUT_F32>(st, A, lda, B, ldb, M, N, K, splitbuf, splitbuf_floats, o); break;
    case OUT_RELU: gemm_out<OUT_RELU>(st, A, lda, B, ldb, M, N, K, splitbuf, splitbuf_floats, o); break;
    case OUT_MASK: gemm_out<OUT_MASK>(st, A, lda, B, ldb, M, N, K, splitbuf, splitbuf_floats, o); break;
    case OUT_MSE: gemm_out<OUT_MSE>(st, A, lda, B, ldb, M, N, K, splitbuf, splitbuf_floats, o); break;
    case OUT_ADAM: gemm_out<OUT_ADAM>(st, A, lda, B, ldb, M, N, K, splitbuf, splitbuf_floats, o); break;
    default: return -1;
  }
  return 0;
}

__global__ void k_split_reduce(const float *__restrict__ part, int splits,
                               long long n, float *__restrict__ out) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = part[i];
  for (int z = 1; z < splits; z++) s += part[(long long)z * n + i];
  out[i] = s;
}

int gemm_skinny(hipStream_t st, const bf16 *A, int lda, const bf16 *B, int ldb,
                float *C, int M, int N, int K, float *splitbuf,
                size_t splitbuf_floats, int min_blocks) {
  if (!gemm_shape_ok(GEMM_CFG_SKINNY, M, N, K, lda, ldb)) return -1;
  const int gm = M / 16, gn = N / 128;
  const long long mn = (long long)M * N;
  const int splits = splitbuf ? gemm_splits(gm * gn, mn, K, splitbuf_floats, min_blocks) : 1;
  GemmOut o{};
  o.outF = splits > 1 ? splitbuf : C;
  hipLaunchKernelGGL((k_gemm_nt<GEMM_SKINNY, false, OUT_F32>), dim3(gn, gm, splits), dim3(256),
                     0, st, A, lda, B, ldb, M, N, K / splits, 1, splits > 1 ? mn : 0, o);
  if (splits > 1)
    hipLaunchKernelGGL(k_split_reduce, dim3((unsigned)((mn + 255) / 256)),
                       dim3(256), 0, st, splitbuf, splits, mn, C);
  return 0;
}

// ---- BF16 copies ----
// out = bf16(op(Z)) and outT = its transpose (either may be null); op: RELU
// max(z,0); PLAIN z.  32x32 tiles through LDS.
__global__ void k_epi(const float *__restrict__ Z, int M, int N, int mode,
                      bf16 *__restrict__ out, bf16 *__restrict__ outT) {
  __shared__ float tile[32][33];
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x, ty = threadIdx.y;  // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const int i = by + r, j = bx + tx;
    float v = 0.f;
    if (i < M && j < N) {
      const long long idx = (long long)i * N + j;
      v = Z[idx];
      if (mode == EPI_RELU) v = v > 0.f ? v : 0.f;
      if (out) out[idx] = (bf16)v;
    }
    tile[r][tx] = v;
  }
  if (!outT) return;
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int j = bx + r, i = by + tx;
    if (i < M && j < N) outT[(long long)j * M + i] = (bf16)tile[tx][r];
  }
}

void epilogue(hipStream_t st, const float *Z, int M, int N, int mode, bf16 *out,
              bf16 *outT) {
  hipLaunchKernelGGL(k_epi, dim3((N + 31) / 32, (M + 31) / 32), dim3(32, 8), 0,
                     st, Z, M, N, mode, out, outT);
}

// ---- encoder: Conv1d(1 -> C, width T, stride S), zero padding, ReLU ----
// Output position p reads nodes S*p - (T-S)/2 + t, t < T; feature p*C + c.
// Row b of the batch is row idx[b] of X (row b without idx), rows >= B are
// zero.  Block = 32 rows x 8 positions x 8 channels, a thread one row and
// position with its taps read once for the 8 channels; the transposed copy
// goes through LDS.
constexpr int kConvCB = 8, kConvTB = 64;  // channels, taps staged at a time

__global__ __launch_bounds__(256) void k_conv_fwd(
    const float *__restrict__ X, const int *__restrict__ idx, int B, int M, int nk,
    const float *__restrict__ Wc, int C, int T, int S, int P0, bf16 *__restrict__ H0,
    bf16 *__restrict__ H0T) {
  __shared__ bf16 ht[32][8 * kConvCB + 2];
  __shared__ float ws[kConvTB][kConvCB];
  const int F0 = P0 * C, tid = threadIdx.x;
  const int p0 = blockIdx.x * 8, b0 = blockIdx.y * 32, c0 = blockIdx.z * kConvCB;
  const int p = p0 + (tid & 7), b = b0 + (tid >> 3), nc = min(kConvCB, C - c0);
  const bool in = b < B && p < P0;
  const int x0 = S * p - (T - S) / 2;
  const float *x = X + (long long)(in ? (idx ? idx[b] : b) : 0) * nk;
  float acc[kConvCB];
#pragma unroll
  for (int c = 0; c < kConvCB; c++) acc[c] = 0.f;
  for (int t0 = 0; t0 < T; t0 += kConvTB) {
    const int nt = min(kConvTB, T - t0);
    __syncthreads();
    for (int e = tid; e < nt * kConvCB; e += 256) {
      const int t = e / kConvCB, c = e % kConvCB;
      if (c < nc) ws[t][c] = Wc[(c0 + c) * T + t0 + t];
    }
    __syncthreads();
    for (int t1 = 0; t1 < nt; t1 += 8) {
      float xt[8];
#pragma unroll
      for (int u = 0; u < 8; u++) xt[u] = x[min(max(x0 + t0 + t1 + u, 0), nk - 1)];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int q = x0 + t0 + t1 + u;
        if (in && t1 + u < nt && q >= 0 && q < nk)
#pragma unroll
          for (int c = 0; c < kConvCB; c++) acc[c] = acc[c] + ws[t1 + u][c] * xt[u];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < kConvCB; c++) {
    const bf16 h = (bf16)(acc[c] > 0.f ? acc[c] : 0.f);
    ht[tid >> 3][(tid & 7) * kConvCB + c] = h;
    if (c < nc && b < M && p < P0) H0[(long long)b * F0 + p * C + c0 + c] = h;
  }
  if (!H0T) return;
  __syncthreads();
  for (int e = tid; e < 32 * 8 * kConvCB; e += 256) {
    const int r = e & 31, f = e >> 5, q = p0 + f / kConvCB, c = f % kConvCB;
    if (c < nc && q < P0 && b0 + r < M)
      H0T[(long long)(q * C + c0 + c) * M + b0 + r] = ht[r][f];
  }
}

void conv_forward(hipStream_t st, const float *X, const int *idx, int B, int M, int nk,
                  const float *Wc, int C, int T, int S, int P0, bf16 *H0, bf16 *H0T) {
  hipLaunchKernelGGL(k_conv_fwd,
                     dim3((P0 + 7) / 8, (M + 31) / 32, (C + kConvCB - 1) / kConvCB),
                     dim3(256), 0, st, X, idx, B, M, nk, Wc, C, T, S, P0, H0, H0T);
}

// dWc[c][t] = sum_b sum_p dZ0[b][p*C+c] * x[b][S*p - (T-S)/2 + t] over the
// rows b < B; one block per (c, t), each thread every 256th term in order with
// the loads of kConvAhead terms in flight, then a fixed-order tree.  With
// Adam coefficients (w given) the weight is updated, else gWc receives the
// gradient.  One more block sums the loss's partial sums.  54 us with one term
// in flight and the rows of padding, 17.5 us now (64 blocks, 160 rows of 128
// positions).
constexpr int kConvAhead = 16;

__global__ __launch_bounds__(256) void k_conv_bwd(
    const float *__restrict__ X, const int *__restrict__ idx, int B, int nk,
    const float *__restrict__ dZ0, int C, int T, int S, int P0, float *__restrict__ gWc,
    float *__restrict__ w, float *__restrict__ m, float *__restrict__ v, AdamCoef k,
    const double *__restrict__ partial, int npart, double scale, double *__restrict__ loss) {
  __shared__ double redd[256];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x == C * T) {
    double s = 0.0;
    for (int i = tid; i < npart; i += 256) s += partial[i];
    redd[tid] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
      if (tid < h) redd[tid] += redd[tid + h];
      __syncthreads();
    }
    if (tid == 0) *loss = redd[0] * scale;
    return;
  }
  float *const red = reinterpret_cast<float *>(redd);
  const int c = blockIdx.x / T, t = blockIdx.x % T;
  const int F0 = P0 * C, n = B * P0, q0 = t - (T - S) / 2;
  const int db = 256 / P0, dp = 256 % P0;
  int b = tid / P0, p = tid % P0;
  float acc = 0.f;
  for (int i = tid; i < n; i += 256 * kConvAhead) {
    // every index clamped into range, so that the loads need no branches
    float z[kConvAhead], x[kConvAhead];
    int row[kConvAhead], at[kConvAhead];
    bool in[kConvAhead];
#pragma unroll
    for (int u = 0; u < kConvAhead; u++) {
      const int q = S * p + q0, bb = min(b, B - 1);
      in[u] = b < B && q >= 0 && q < nk;
      at[u] = min(max(q, 0), nk - 1);
      z[u] = dZ0[(long long)bb * F0 + p * C + c];
      row[u] = idx ? idx[bb] : bb;
      b += db;
      p += dp;
      if (p >= P0) {
        p -= P0;
        b++;
      }
    }
#pragma unroll
    for (int u = 0; u < kConvAhead; u++) x[u] = X[(long long)row[u] * nk + at[u]];
#pragma unroll
    for (int u = 0; u < kConvAhead; u++)
      if (in[u]) acc = acc + z[u] * x[u];
  }
  red[tid] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) red[tid] = red[tid] + red[tid + s];
    __syncthreads();
  }
  if (tid != 0) return;
  const int i = c * T + t;
  if (w) {
    float wi = w[i], mi = m[i], vi = v[i];
    adam_step(k, red[0], wi, mi, vi);
    w[i] = wi;
    m[i] = mi;
    v[i] = vi;
  } else {
    gWc[i] = red[0];
  }
}

void conv_backward(hipStream_t st, const float *X, const int *idx, int B, int nk,
                   const float *dZ0, int C, int T, int S, int P0, float *gWc, float *w,
                   float *m, float *v, const AdamCoef &k, const double *partial, int npart,
                   double scale, double *loss) {
  hipLaunchKernelGGL(k_conv_bwd, dim3(C * T + 1), dim3(256), 0, st, X, idx, B, nk, dZ0, C, T,
                     S, P0, gWc, w, m, v, k, partial, npart, scale, loss);
}

}  // namespace nn
}  // namespace qdeq
