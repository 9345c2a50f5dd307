// Expert products of a decode step (at most 256 routed pairs), on fragment-major expert weights (ops.gemm.frag_weight): two launches,
// no routing launch, no row tiles.
//
// Bound: a step of 12 tokens runs every expert on two to four rows, so its time is the weights' way from the Infinity Cache and what
// stands in front of it.  On the LDS-tiled grouped GEMM that was a route launch of one workgroup (5 us) and 64-row tiles whose loads of
// rows touch 16 lines for the bytes of 8 (15 + 10 us a layer of 8 experts of 1024 x 1024).  Here a wave owns one 16-column tile of one
// expert and the whole of K, streams it as contiguous kilobytes, and finds the expert's pairs itself: 64 ids are a ballot.
// One wave a tile (KS 1): its sum over K is the chain of the grouped GEMM (ascending, one accumulator, same operand order), the same
// bits, for models that need them.  KS 4: four waves of a tile share K and meet in LDS, a quarter of the chain.  A layer of 8 or 9 experts is
// 512 to 1152 workgroups, so what a wave keeps in registers decides whether they run side by side: with three stages and row blocks of
// 64 (180 registers, two workgroups a CU, the rest in a second round) both products of 8 experts took 20.5 us at 12 tokens and 21.0 at
// 24, with two stages and rows by 32 (105 registers, four a CU) 15.9 and 17.2; 9 squared-ReLU experts 18.6 -> 14.8 at 12, 21.5 -> 18.3
// at 24 tokens.  Without conditions before the loads, one launch in a captured graph, 12 tokens, weights from HBM: one wave a tile 8 experts
// 2048 x 1024 11.8 -> 9.5, 1024 x 1024 7.0 -> 5.6; four waves 9 of 1024 x 1024 5.8 -> 5.6, 64 of 2816 x 2048 63.4 -> 62.2.
//
//   moe_decode_kernel<ACT 0>  act[pair] = silu(g) u of x[pair / k], weights paired 8 columns apart
//                    <ACT 1>  act[pair] = relu(x . w)^2
//                    <ACT 2>  y[pair] = act[pair] . w2 in bf16, <ACT 3> kept in f32
// Rows are in pair order, so the sums over a token's experts (moe.hip, seqmix.hip) need no permutation.
#include "common.h"

namespace {
constexpr int MD_PAIRS = 256;
constexpr int MD_TILES = 2;      // column tiles a workgroup of KS 1: the 64 x 9 waves of a 1024-wide layer reach every CU

// 32 k of a tile's weights; past the buffer's last k zeros that cost no traffic
__device__ __forceinline__ bf16x8 md_w(__amdgpu_buffer_rsrc_t r, int k) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, (unsigned)k * 32 + (threadIdx.x & 63) * 16, 0, 0));
}

template <int ACT, int MT, int KS>
__device__ __forceinline__ void expert_rows(const u16* __restrict__ x, long ldx, int div, __amdgpu_buffer_rsrc_t wt, int kb, int K,
                                            const int* list, int row0, int n, int c0, void* __restrict__ out, long ldo,
                                            const bf16x8 (&w0)[4], float (*s_acc)[KS > 1 ? 32 : 1][17]) {      // k in [kb, K)
  const int lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
  // no load stands behind a condition (rows past n read the last one's, k past the end nothing or the last step's; neither is used):
  // where ways with and without a load meet the compiler waits for all loads in flight
  const u16* xr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = x + (long)(list[min(row0 + 16 * m + r16, n - 1)] / div) * ldx + 8 * g;
  constexpr int U = MT > 2 || (KS > 1 && MT > 1) ? 2 : 4;
  const int klast = max(K - 32, 0);
  struct Stage { bf16x8 w[U]; uint4 x[U][MT]; };
  auto load = [&](Stage& st, int k0, int first) {      // `first`: the stage's place among the weights loaded ahead (-1: not there)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      st.w[u] = first >= 0 ? w0[first + u] : md_w(wt, k0 + 32 * u);
#pragma unroll
      for (int m = 0; m < MT; ++m) st.x[u][m] = ld16(xr[m] + min(k0 + 32 * u, klast));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const Stage& st, int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + 32 * u >= K) break;      // (uniform)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, st.x[u][m]), st.w[u], acc[m], 0, 0, 0);
    }
  };
  Stage A, B;
  load(A, kb, 0);
  // A quarter of K is two stages or little more: stages that do not exist are not asked for (they reach no memory, but pass through the caches'
  // pipe like any other), and ways part only where nothing of theirs meets in flight.  64 experts of 2048 x 1408, 11 and 16 steps a quarter, 24
  // to 64 tokens 3 % longer than with loads behind conditions before, now 1 to 5 % shorter; of 1024 x 512 64 tokens 45.5 -> 41.2 us
  if constexpr (KS > 1) {
    if (kb + 32 * U >= K) compute(A, kb);
    else {
      load(B, kb + 32 * U, U == 2 ? 2 : -1);
      int k0 = kb;
      for (; k0 + 96 * U < K; k0 += 64 * U) {
        compute(A, k0);
        load(A, k0 + 64 * U, -1);
        compute(B, k0 + 32 * U);
        load(B, k0 + 96 * U, -1);
      }
      compute(A, k0);
      if (k0 + 64 * U < K) {
        load(A, k0 + 64 * U, -1);
        compute(B, k0 + 32 * U);
        compute(A, k0 + 64 * U);
      } else compute(B, k0 + 32 * U);
    }
  } else {
    load(B, kb + 32 * U, U == 2 ? 2 : -1);
    int k0 = kb;
    Stage C;      // two stages ahead of the one that is multiplied
    load(C, k0 + 64 * U, -1);
    for (; k0 + 96 * U < K; k0 += 96 * U) {
      compute(A, k0);
      load(A, k0 + 96 * U, -1);
      compute(B, k0 + 32 * U);
      load(B, k0 + 128 * U, -1);
      compute(C, k0 + 64 * U);
      load(C, k0 + 160 * U, -1);
    }
    compute(A, k0);
    compute(B, k0 + 32 * U);
    compute(C, k0 + 64 * U);
  }
  auto put = [&](int row, int c, float a, float u) {
    if (row >= n) return;
    if constexpr (ACT == 0) {
      const float gv = bf2f(f2bf(a)), uv = bf2f(f2bf(u));
      reinterpret_cast<u16*>(out)[list[row] * ldo + c0 / 2 + c] = f2bf(gv / (1.f + __expf(-gv)) * uv);
    } else {
      const float rl = fmaxf(a, 0.f);
      if constexpr (ACT == 3) reinterpret_cast<float*>(out)[list[row] * ldo + c0 + c] = a;
      else reinterpret_cast<u16*>(out)[list[row] * ldo + c0 + c] = f2bf(ACT == 1 ? rl * rl : a);
    }
  };
  if constexpr (KS > 1) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __syncthreads();      // (a second pass of rows: the first one's sums are read)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) s_acc[wave][16 * m + 4 * g + r][r16] = acc[m][r];
    __syncthreads();
    constexpr int NC = ACT == 0 ? 8 : 16;
    for (int i = threadIdx.x; i < 16 * MT * NC; i += 64 * KS) {
      const int row = i / NC, c = i % NC;
      auto sum = [&](int c) { return (s_acc[0][row][c] + s_acc[1][row][c]) + (s_acc[2][row][c] + s_acc[3][row][c]); };
      put(row0 + row, c, sum(c), ACT == 0 ? sum(c + 8) : 0.f);
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float u = ACT == 0 ? lane_xor(acc[m][r], 8) : 0.f;
      if (ACT != 0 || r16 < 8) put(row0 + 16 * m + 4 * g + r, r16, acc[m][r], u);
    }
}

template <int ACT, int KS>
__global__ void __launch_bounds__(KS > 1 ? 64 * KS : 64 * MD_TILES, KS > 1 ? 4 : 1) moe_decode_kernel(const u16* __restrict__ x, long ldx, int div, const int* __restrict__ ids, int P,
                                                                   int E, const u16* __restrict__ w, int N, int K, void* __restrict__ out,
                                                                   long ldo) {
  constexpr int WV = KS > 1 ? KS : MD_TILES;
  __shared__ int s_list[WV][MD_PAIRS];
  __shared__ float s_acc[KS > 1 ? KS : 1][KS > 1 ? 32 : 1][17];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = blockIdx.y, tile = KS > 1 ? blockIdx.x : blockIdx.x * MD_TILES + wave;
  if (tile * 16 >= N) return;      // (KS 1: no barrier below)
  const int kq = KS > 1 ? (K / KS + 31) & ~31 : K, kb = KS > 1 ? min(K, wave * kq) : 0, ke = min(K, kb + kq);
  const __amdgpu_buffer_rsrc_t wt = make_rsrc(w + ((long)e * (N / 16) + tile) * 16 * K, (unsigned)ke * 32);
  // The ids first: loads come back in order, and behind the weights the list waited for those (64 experts of 1024 x 512, 64 tokens of 4, 50.1 -> 45.5 us)
  int id[MD_PAIRS / 64];
#pragma unroll
  for (int b = 0; b < MD_PAIRS / 64; ++b) id[b] = ids[min(64 * b + lane, P - 1)];
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 w0[4];
  auto first = [&] {
#pragma unroll
    for (int u = 0; u < 4; ++u) w0[u] = md_w(wt, kb + 32 * u);
  };
  // The first weights are under way while the ids come, unless many experts have no pair and would stream them for nothing.  us always
  // ahead / here: two tokens of 4 of 64 experts of 2048 x 1408 74 / 34, 16 tokens 141 / 124, 32 (two pairs an expert) 173 / 169, 48 180 / 180; of 1024
  // x 512 16 tokens 36.6 / 31.0, 32 39.8 / 39.5, and 64 with none ahead 42.9, ahead 41.2
  const bool early = P > 2 * E;
  if (early) first();
  int* list = s_list[wave];
  int n = 0;
#pragma unroll
  for (int b = 0; b < MD_PAIRS / 64; ++b) {
    const int p = 64 * b + lane;
    const bool mine = p < P && min(max(id[b], 0), E - 1) == e;
    const unsigned long long m = __ballot(mine);
    if (mine) list[n + __popcll(m & ((1ull << lane) - 1ull))] = p;
    n += __popcll(m);
  }
  if (n == 0) return;
  if (!early) first();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");      // the list is the wave's own: in order through LDS
  __builtin_amdgcn_wave_barrier();
  if (n <= 16) expert_rows<ACT, 1, KS>(x, ldx, div, wt, kb, ke, list, 0, n, tile * 16, out, ldo, w0, s_acc);
  else if (n <= 32) expert_rows<ACT, 2, KS>(x, ldx, div, wt, kb, ke, list, 0, n, tile * 16, out, ldo, w0, s_acc);
  else if constexpr (KS > 1)
    for (int r = 0; r < n; r += 32) expert_rows<ACT, 2, KS>(x, ldx, div, wt, kb, ke, list, r, n, tile * 16, out, ldo, w0, s_acc);
  else
    for (int r = 0; r < n; r += 64) expert_rows<ACT, 4, KS>(x, ldx, div, wt, kb, ke, list, r, n, tile * 16, out, ldo, w0, s_acc);
}
}  // namespace

// act 0 SwiGLU (w paired, N = 2 I columns, out bf16 [P, I]), 1 squared ReLU (out bf16), 2 plain bf16, 3 plain f32.  w: per expert
// [N / 16][K / 32][64][8]; row of pair p: x + (p / div) ldx; ids [P], P <= 256; ks 1 (the
// grouped GEMM's bits) or 4 waves a tile.
extern "C" int dllm_moe_decode(const void* x, long ldx, int div, const int* ids, int P, int E, const void* w, int N, int K, int act,
                               int ks, void* out, long ldo, hipStream_t st) {
  if (P < 1 || P > MD_PAIRS || E < 1 || N < 16 || N % 16 || K < 32 || K % 32 || div < 1 || ldx % 8 || (act == 0 && N % 32)) return -1;
#define MD_GO(A)                                                                                                                        \
  if (ks == 4)                                                                                                                          \
    hipLaunchKernelGGL((moe_decode_kernel<A, 4>), dim3(N / 16, E), dim3(256), 0, st, (const u16*)x, ldx, div, ids, P, E, (const u16*)w, N, K, out, ldo); \
  else                                                                                                                                  \
    hipLaunchKernelGGL((moe_decode_kernel<A, 1>), dim3((N / 16 + MD_TILES - 1) / MD_TILES, E), dim3(64 * MD_TILES), 0, st, (const u16*)x, ldx, div, \
                       ids, P, E, (const u16*)w, N, K, out, ldo)
  switch (act) {
    case 0: MD_GO(0); break;
    case 1: MD_GO(1); break;
    case 2: MD_GO(2); break;
    case 3: MD_GO(3); break;
    default: return -2;
  }
#undef MD_GO
  return (int)hipGetLastError();
}
