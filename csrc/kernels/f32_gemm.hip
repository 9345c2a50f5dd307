// Projections of up to 16 rows of an f32 model:  Y = X[M, K] . W[N, K]^T [-> erf-GELU],  f32 in, f32 matrix instructions.
//
// At these sizes a product is bound by a few loads' latency, not by its flops or its weights: 16 columns of 512 k are four loads of a
// wave.  So a workgroup takes 16 columns and all rows, its eight waves share K with up to eight steps of 16 k in flight each, and meet
// in LDS; W is kept as [N / 16][K / 16][64 lanes][4] (ops.gemm.frag_weight), a wave's load is 1 KB in a row.  mfma_f32_16x16x4 takes
// one float a lane and operand; lane 16 g + r holds k = 16 s + 4 g + j of row r in component j, so four instructions on the four
// components multiply 16 k, both operands in the same order.
// 2 rows, N x K 512 x 512 / 2048 x 512 / 1536 x 1024 / 512 x 2048 / 2048 x 2048 / 32000 x 512: 2.9 / 3.5 / 4.1 / 6.0 / 6.2 / 12.7 us
// against the vendor GEMM's 4.3 / 5.9 / 8.2 / 8.4 / 9.7 / 15.1 (16 rows 3.4 / 3.9 / 5.2 / 8.0 / 8.6 / 14.5 against 4.4 / 5.9 / 8.2 / 8.4
// / 10.1 / 16.5); 4 or 16 waves lie up to a fifth behind.  Eight partial sums of K / 8 terms lie nearer to 64 bits, too: 512 k 1.5e-7
// against 2.0e-7, 2048 k 2.9e-7 against 4.1e-7.  1024 x 4096 is even at 2 rows (10.2) and behind at 16 (14.7 against 10.8): longer K and
// more rows (512 x 2048 on 24: 10.9 against 8.4) stay with the vendor.
#include "common.h"

namespace {
enum { FG_PLAIN = 0, FG_GELU = 5 };

constexpr int NW = 8;

template <int EPI>
__global__ void __launch_bounds__(64 * NW) f32_gemm_kernel(const float* __restrict__ X, long ldx, const float* __restrict__ W,
                                                           float* __restrict__ Y, long ldy, int M, int N, int K) {
  constexpr int KS = 8, RS = 20;      // LDS rows of 16 + 4 floats reach every bank
  __shared__ __attribute__((aligned(16))) float red[NW][16][RS];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g = lane >> 4;
  const int steps = K / 16, per = (steps + NW - 1) / NW, s0 = min(steps, w * per), s1 = min(steps, s0 + per);
  const float* wr = W + (long)blockIdx.x * 16 * K + 4 * lane;
  const float* xr = X + (long)min(lr, M - 1) * ldx + 4 * g;      // rows past M repeat the last and are dropped
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += KS) {
    f32x4 wf[KS], xf[KS];
#pragma unroll
    for (int u = 0; u < KS; ++u)
      if (s + u < s1) {
        wf[u] = *reinterpret_cast<const f32x4*>(wr + (long)(s + u) * 256);
        xf[u] = *reinterpret_cast<const f32x4*>(xr + 16 * (s + u));
      }
#pragma unroll
    for (int u = 0; u < KS; ++u)
      if (s + u < s1)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xf[u][j], wf[u][j], acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[w][4 * g + i][lr] = acc[i];
  __syncthreads();
  const int row = threadIdx.x >> 2, c = 4 * (threadIdx.x & 3), col = blockIdx.x * 16 + c;
  if (row >= M) return;               // M <= 16 rows of four threads each: the first wave
  f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][row][c]);
#pragma unroll
  for (int j = 1; j < NW; ++j) v += *reinterpret_cast<const f32x4*>(&red[j][row][c]);
  if (EPI == FG_GELU)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = 0.5f * v[i] * (1.f + erff(v[i] * 0.70710678118654752f));
  float* y = Y + (long)row * ldy + col;
  if (col + 4 <= N && (ldy & 3) == 0) *reinterpret_cast<f32x4*>(y) = v;
  else
    for (int i = 0; i < 4; ++i)
      if (col + i < N) y[i] = v[i];
}

}  // namespace

// W: ops.gemm.frag_weight's [ceil(N / 16)][K / 16][64][4].  X rows of a multiple of 4 floats, 16-byte aligned; Y 16-byte aligned.
extern "C" int dllm_f32_gemm(const float* X, long ldx, const float* W, float* Y, long ldy, int M, int N, int K, int epi, hipStream_t st) {
  if (M < 1 || M > 16 || N < 1 || K < 16 || K % 16 || ldx % 4 || (M > 1 && (ldx < K || ldy < N)) ||
      (((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) & 15))
    return -1;
  const dim3 g((N + 15) / 16), b(64 * NW);
  if (epi == FG_PLAIN) hipLaunchKernelGGL((f32_gemm_kernel<FG_PLAIN>), g, b, 0, st, X, ldx, W, Y, ldy, M, N, K);
  else if (epi == FG_GELU) hipLaunchKernelGGL((f32_gemm_kernel<FG_GELU>), g, b, 0, st, X, ldx, W, Y, ldy, M, N, K);
  else return -2;
  return (int)hipGetLastError();
}
