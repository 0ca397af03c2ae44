// Batched fp32 products on few rows: Y[b] = A[b] W[b]^T (+ bias[b]) (+ R[b]), the node-side linears of a
// small system (a few dozen to a few hundred atoms, one weight per coefficient, K = 128 or 256).
//
// The 128-row tiles of gemm.hip put one workgroup on each batch entry there, and its 8 chunks of
// load, split, barrier and product run one after the other: 12 us at 54 rows whatever the rate of
// the matrix cores.  Here a workgroup owns 16 rows and 128 columns: the A rows in LDS whole, each of
// the eight waves 16 columns, its weights loaded straight into the B operands of
// v_mfma_f32_16x16x4_f32 with all loads of 128 k in flight at once, issued before the A tile arrives.
// Nothing is scaled or split, and each output is four sums of K / 4 exact products added at the end.
// The price, 1/16 of the fp16 rate and the weight read once per 16 rows, is why many rows stay on the
// 128-row tiles (use_rows16 in gemm.hip, with the figures).  An atom-wise feed-forward block of 54 atoms
// (C = 128, lmax 2, forward and backward) takes 40 us with it, 78 without.
#include "fu_vec.h"

namespace fu {
namespace r16 {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int ROWS = 16, COLS = 128, KC = 128;

// 16 rows of A from n0 on (zeros past M), KB columns from k0 on, into LDS rows of LD floats
template <int LD>
__device__ __forceinline__ void stage_rows(const float* A, int64_t lda, int64_t n0, int64_t M, int k0, int kb, float* at) {
  for (int i = threadIdx.x; i < ROWS * (kb / 4); i += 512) {
    const int row = i / (kb / 4), c = 4 * (i - row * (kb / 4));
    const int64_t n = n0 + row;
    st4(at + row * LD + c, n < M ? ld4(A + n * lda + k0 + c) : make_float4(0.f, 0.f, 0.f, 0.f));
  }
}

__global__ __launch_bounds__(512) void linear_rows16_kernel(
    const float* __restrict__ A, int64_t lda, int64_t sA, const float* __restrict__ W, int64_t ldw, int64_t sW,
    const float* __restrict__ bias, int64_t sBias, int32_t bias_batches, const float* R, int64_t ldr, int64_t sR,
    float* Y, int64_t ldy, int64_t sY, int64_t M, int32_t N, int32_t K) {
  constexpr int LD = KC + 4;
  __shared__ __attribute__((aligned(16))) float at[ROWS * LD];
  const int64_t b = blockIdx.y, n0 = (int64_t)blockIdx.x * ROWS;
  A += b * sA;
  Y += b * sY;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int col = (int)blockIdx.z * COLS + (int)(threadIdx.x >> 6) * 16 + r;
  const bool live = col < N;   // N is a multiple of 16: whole waves
  // this lane's column of W, k 8 g .. 8 g + 7 of every 32 (a dead wave reads column 0)
  const float* w = W + b * sW + (int64_t)(live ? col : 0) * ldw + 8 * g;
  // four sums per output, one per k mod 4: no product waits for the one before
  floatx4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = 0; k0 < K; k0 += KC) {
    const int kb = K - k0 < KC ? K - k0 : KC;   // a multiple of 32
    float4 f[KC / 32][2];
#pragma unroll
    for (int j = 0; j < KC / 32; ++j) {   // past K: the first piece again, not used
      const float* p = w + k0 + (32 * j < kb ? 32 * j : 0);
      f[j][0] = ld4(p);
      f[j][1] = ld4(p + 4);
    }
    if (k0 > 0) __syncthreads();
    stage_rows<LD>(A, lda, n0, M, k0, kb, at);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < KC / 32; ++j) {
      if (32 * j >= kb) break;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float4 a = ld4(at + r * LD + 32 * j + 8 * g + 4 * h);
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32((&a.x)[t], (&f[j][h].x)[t], acc[t], 0, 0, 0);
      }
    }
  }
  if (!live) return;
  const float add = bias != nullptr && b < bias_batches ? bias[b * sBias + col] : 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t n = n0 + 4 * g + i;
    if (n >= M) continue;
    float y = (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]) + add;
    if (R) y += R[b * sR + n * ldr + col];   // R may be Y: this thread's own element
    Y[n * ldy + col] = y;
  }
}

}  // namespace r16

void launch_linear_rows16(const float* A, int64_t lda, int64_t sA, const float* W, int64_t ldw, int64_t sW,
                          const float* bias, int64_t sBias, int32_t bias_batches, const float* R, int64_t ldr,
                          int64_t sR, float* Y, int64_t ldy, int64_t sY, int64_t M, int32_t N, int32_t K,
                          int32_t batch, hipStream_t s) {
  hipLaunchKernelGGL(r16::linear_rows16_kernel, dim3(cdiv(M, r16::ROWS), (unsigned)batch, cdiv(N, r16::COLS)), dim3(512),
                     0, s, A, lda, sA, W, ldw, sW, bias, sBias, bias_batches, R, ldr, sR, Y, ldy, sY, M, N, K);
}

}  // namespace fu
