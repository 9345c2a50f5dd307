// Projections of up to 16 rows of an f32 model:  Y = X[M, K] . W[N, K]^T [-> erf-GELU],  f32 in, f32 matrix instructions.
//
// At these sizes a product is bound by a few loads' latency, not by its flops or its weights: 16 columns of 512 k are four loads of a
// wave.  So a workgroup takes 16 columns and all rows, its eight waves share K with up to eight steps of 16 k in flight each, and meet
// in LDS; W is kept as [N / 16][K / 16][64 lanes][4] (ops.gemm.frag_weight), a wave's load is 1 KB in a row.  mfma_f32_16x16x4 takes
// one float a lane and operand; lane 16 g + r holds k = 16 s + 4 g + j of row r in component j, so four instructions on the four
// components multiply 16 k, both operands in the same order.
// 16 rows, N x K 512 x 512 / 2048 x 512 / 1536 x 1024 / 512 x 2048 / 2048 x 2048 / 32000 x 512: 3.4 / 3.9 / 5.2 / 8.0 / 8.6 / 14.5 us
// against the vendor GEMM's 4.4 / 5.9 / 8.2 / 8.4 / 10.1 / 16.5; 4 or 16 waves lie up to a fifth behind.  Eight partial sums of K / 8 terms lie
// nearer to 64 bits, too: 512 k 1.5e-7 against 2.0e-7, 2048 k 2.9e-7 against 4.1e-7.  1024 x 4096 is behind at 16 (14.7 against 10.8):
// longer K and more rows (512 x 2048 on 24: 10.9 against 8.4) stay with the vendor.
// Up to eight rows are another kernel: there the 16 x 16 product, most of it rows that do not exist, is what a long K takes (256 steps
// of 4096 k are 3.7 us of a CU's matrix cores), and then the loads of X, sixteen pieces of 16 lines for what is two.
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

// The same of at most 4 RB rows: mfma_f32_4x4x1 is sixteen products of 4 x 4 x 1 in a quarter of the time.  Its block of lanes 16 g + 4 q ..
// + 3 takes columns 4 q .. + 3 at the k of group g from the weights as they lie, against four rows at that k; the four groups' sums meet
// ahead of the waves'.  X is read in rows, KS steps at a time, and goes round to the lanes through a piece of LDS that is the wave's own
// (pieces of a k 16 bytes off the power of two: at eight rows of 1024 x 1024 4.4 us without, here 4.0).  us, the kernel above / here (the
// vendor's): 2 rows 512 x 512 2.96 / 2.68 (4.4), 2048 x 512 3.4 / 3.1 (5.8), 1024 x 1024 4.1 / 3.5 (8.1), 1024 x 2048 6.2 / 4.4 (8.5), 2048 x
// 2048 6.1 / 5.0 (8.7), 1024 x 4096 10.2 / 6.1 (10.1), 2048 x 8192 22.3 / 18.1 (22.7), 32000 x 1024 25.1 / 23.0 (32.4); 8 rows 2048 x 512 3.6 /
// 3.5, 1024 x 1024 4.5 / 4.0, 2048 x 2048 7.4 / 5.5, 1024 x 4096 12.3 / 7.5 (10.1).  Sums of K / 64 terms with sixteen waves, K / 32 with
// eight (K up to 512, and the weights of 64 MB and more): with sixteen 1.4e-7 from 64 bits at 2048 k, 3.0e-7 above.
template <int EPI, int RB, int NWV, int KS>
__global__ void __launch_bounds__(64 * NWV) f32_few_kernel(const float* __restrict__ X, long ldx, const float* __restrict__ W, float* __restrict__ Y,
                                                           long ldy, int M, int N, int K) {
  constexpr int RS = 20;
  __shared__ __attribute__((aligned(16))) float red[NWV][4 * RB][RS];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g = lane >> 4;
  const int steps = K / 16, per = (steps + NWV - 1) / NWV, s0 = min(steps, w * per), s1 = min(steps, s0 + per);
  const float* wr = W + (long)blockIdx.x * 16 * K + 4 * lane;
  __shared__ __attribute__((aligned(16))) f32x4 sx[NWV][KS * 4 * (4 * RB + 1)];
  f32x4 acc[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int R = 4 * RB, XL = KS * 4 * R / 64, PR = KS * 4;      // rows, 16-byte pieces of X a lane, pieces a row
  const float* xr[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) xr[i] = X + (long)min((lane + 64 * i) / PR, M - 1) * ldx + 4 * ((lane + 64 * i) % PR);      // (rows past M repeat the last)
  for (int s = s0; s < s1; s += KS) {
    f32x4 wf[KS], xv[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i)
      if (s + (lane + 64 * i) % PR / 4 < s1) xv[i] = *reinterpret_cast<const f32x4*>(xr[i] + 16 * s);
#pragma unroll
    for (int u = 0; u < KS; ++u)
      if (s + u < s1) wf[u] = *reinterpret_cast<const f32x4*>(wr + (long)(s + u) * 256);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < XL; ++i) sx[w][((lane + 64 * i) % PR) * (R + 1) + (lane + 64 * i) / PR] = xv[i];
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < KS; ++u)
      if (s + u < s1) {
        f32x4 xf[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) xf[b] = sx[w][(4 * u + g) * (R + 1) + 4 * b + (lane & 3)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int b = 0; b < RB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_4x4x1f32(xf[b][j], wf[u][j], acc[b], 0, 0, 0);
      }
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = lane_add(lane_add(acc[b][i], 16), 32);
      if (g == 0) red[w][4 * b + i][lr] = v;
    }
  __syncthreads();
  const int row = threadIdx.x >> 2, c = 4 * (threadIdx.x & 3), col = blockIdx.x * 16 + c;
  if (row >= M) return;
  f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][row][c]);
#pragma unroll
  for (int j = 1; j < NWV; ++j) v += *reinterpret_cast<const f32x4*>(&red[j][row][c]);
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
#define FEW(RB, NWV, KS)                                                                                                                    \
  do {                                                                                                                                      \
    if (epi == FG_PLAIN) hipLaunchKernelGGL((f32_few_kernel<FG_PLAIN, RB, NWV, KS>), g, dim3(64 * NWV), 0, st, X, ldx, W, Y, ldy, M, N, K); \
    else hipLaunchKernelGGL((f32_few_kernel<FG_GELU, RB, NWV, KS>), g, dim3(64 * NWV), 0, st, X, ldx, W, Y, ldy, M, N, K);                  \
  } while (0)
  // waves and steps in flight: a short K has no steps for sixteen waves (512 x 512, 2 rows: 2.9 us with them, 2.7 with eight), and a weight from
  // 64 MB on is bound by its stream, which two waves a SIMD with longer loads keep better (4096 x 4096: 15.9 / 14.5)
#define ROWS(RB)                                   \
  do {                                             \
    if (K <= 512) FEW(RB, 8, 4);                   \
    else if (N >= 4096 && K >= 4096) FEW(RB, 8, 8); \
    else FEW(RB, 16, 4);                           \
  } while (0)
  if (epi != FG_PLAIN && epi != FG_GELU) return -2;
  if (M <= 4) ROWS(1);
  else if (M <= 8) ROWS(2);
  else if (epi == FG_PLAIN) hipLaunchKernelGGL((f32_gemm_kernel<FG_PLAIN>), g, b, 0, st, X, ldx, W, Y, ldy, M, N, K);
  else hipLaunchKernelGGL((f32_gemm_kernel<FG_GELU>), g, b, 0, st, X, ldx, W, Y, ldy, M, N, K);
#undef ROWS
#undef FEW
  return (int)hipGetLastError();
}
