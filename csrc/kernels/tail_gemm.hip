// A sublayer's tail in the launch of the product behind it, for steps of up to 16 rows of layer lists with a norm on both sides:
//   x2 = x + rmsnorm(y + bias) * w_post,   h = rmsnorm(x2) * w_next,   out = h . W^T  (or glu_act of it).
//
// A decode step of such a list is bound by its launches, each waiting for the one before it: the residual norm alone is 3.9 us of which
// its bytes (four rows of 1024: 40 KB) are none.  So every workgroup of the product norms all rows itself (6 bytes an entry out of L2,
// 24 KB for four rows, 96 for 16) while its weights are on their way, and the workgroup that a row falls to leaves the updated stream in
// `x2`: a buffer of its own, since the others still read `x`.
//   * 16 waves.  Wave r norms row r: as resadd_norm_vec_kernel (seqmix.hip) does with its 256 threads, a lane standing for four of them, so
//     that a row has the same bits in either launch; the rounded row lies in LDS, 16 bytes off the power of two (fragment reads meet no bank
//     twice).
//   * Product as dgemm_kernel (decode_gemm.hip) with four splits of K a workgroup: fragment-major weights, each wave a sixteenth of K, partial
//     tiles through LDS, the same order of sums.  NT tiles of 16 columns a workgroup: one while a round of workgroups holds them, else two.
// us in a captured graph, width 1024, two launches / here: 1088 columns 1 row 6.1 / 3.9, 4 rows 6.2 / 3.9, 8 6.4 / 4.7, 16 6.8 / 6.3; 3136 columns
// 6.5 / 4.2, 6.5 / 4.1, 6.8 / 4.8, 7.0 / 6.4; 5632 gated 8.4 / 4.9, 8.5 / 5.2, 9.3 / 5.9, 9.3 / 7.8; 8192 7.5 / 5.0, 7.6 / 5.5, 7.8 / 5.7, 7.9 / 7.3
// (two rows a SIMD and more add their arithmetic, 0.2 us a row: widths up to 512 win with up to 12 rows, ops.gemm.tail_wins; 3136 columns of 512 1 row 5.6 /
// 3.8, 8 6.0 / 4.8, 12 6.1 / 5.5, of 768 5.8 / 4.0, 6.4 / 4.8, 16 6.7 / 6.4).
#include "common.h"

namespace {
struct TailArgs {
  const u16* y;
  long ldy;
  const float *x, *w_post, *w_next, *bias;      // bias null: none
  float* x2;
  float eps;
  const u16* W;
  u16* out;
  long ldo;
  int M, N, K;
  const float* act_bias;      // GLU: over the gate columns, then the up columns (null: none)
  int mode;                   // glu_act's
  float limit, alpha;
};

constexpr int WV = 16, MR = 16, MAX_K = 1024, PITCH = MAX_K + 8;

__device__ __forceinline__ void keep_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The row's sum, with the additions of squares<1> (seqmix.hip) and of block_sum over four waves (common.h): four sums over the lanes at once, a
// lane of a 16-lane row standing for one of them from the second exchange on.
__device__ __forceinline__ float squares(const float4& q) { return fmaf(q.w, q.w, fmaf(q.z, q.z, fmaf(q.y, q.y, q.x * q.x))); }
__device__ __forceinline__ float row_sum(const float* s) {
  auto pair = [](float a, float b) {      // lanes below 32: a of the lane and of the one 32 above; the others: b
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
  };
  const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(pair(s[0], s[2])), __float_as_uint(pair(s[1], s[3])), false, false);
  float v = __uint_as_float(t[0]) + __uint_as_float(t[1]);      // rows of 16 lanes: s[0], s[1], s[2], s[3]
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) v = lane_add(v, o);
  float r = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) r += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), 16 * j));
  return r;
}

template <int NT, bool GLU>
__global__ void __launch_bounds__(64 * WV) tail_gemm_kernel(TailArgs a) {
  constexpr int NC = 16 * NT, LD = NC + 4, IPR = GLU ? NC / 8 : NC / 4;      // items a row: four outputs each
  __shared__ __attribute__((aligned(16))) u16 rows[MR * PITCH];
  __shared__ __attribute__((aligned(16))) float part[WV][MR * LD];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, r16 = lane & 15;
  const int tile = blockIdx.x, K = a.K, N = a.N;

  // ---- loads: the wave's row with the norms' weights (a load out of a buffer's range takes its turn in the caches' pipe all the same: with 20 in
  // every wave one row took as long as twelve), then its weights (past its k zeros), then what the epilogue needs
  constexpr unsigned NONE = 0x40000000u;
  const bool mine = wave < a.M;
  uint2 yb[4];
  float4 y[4], v[4], wp[4], wn[4], bi[4];
  if (mine) {
    const float* bp = a.bias ? a.bias : a.w_post;
#pragma unroll
    for (int j = 0; j < 4; ++j) {      // (a vector past the row reads the first and is zero)
      const int c0 = 4 * (64 * j + lane), c = c0 < K ? c0 : 0;
      yb[j] = *reinterpret_cast<const uint2*>(a.y + (long)wave * a.ldy + c);
      v[j] = *reinterpret_cast<const float4*>(a.x + (long)wave * K + c);
      bi[j] = *reinterpret_cast<const float4*>(bp + c);
      wp[j] = *reinterpret_cast<const float4*>(a.w_post + c);
      wn[j] = *reinterpret_cast<const float4*>(a.w_next + c);
    }
  }
  keep_order();
  const int kw = ((K + WV - 1) / WV + 31) & ~31, wk0 = min(K, wave * kw), wk1 = min(K, wk0 + kw);
  constexpr int U = MAX_K / WV / 32;      // k-steps a wave
  const int nt16 = (N + 15) >> 4;
  bf16x8 w[U][NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const __amdgpu_buffer_rsrc_t wt = make_rsrc(a.W + (long)min(tile * NT + n, nt16 - 1) * 16 * K, (unsigned)wk1 * 32);
#pragma unroll
    for (int u = 0; u < U; ++u)
      w[u][n] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wt, (unsigned)((wk0 + 32 * u) * 32 + lane * 16), 0, 2));
  }
  keep_order();
  const int m = threadIdx.x / IPR, q = threadIdx.x % IPR;
  const bool item = m < a.M;
  const int gc = 8 * (tile * NT + q / 2) + 4 * (q & 1);      // GLU: the item's columns
  f32x4 bg = {0.f, 0.f, 0.f, 0.f}, bu = bg;
  if constexpr (GLU) {
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(a.act_bias, a.act_bias ? (unsigned)N * 4 : 0u);
    bg = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, item ? (unsigned)gc * 4 : NONE, 0, 0));
    bu = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, item ? (unsigned)(N / 2 + gc) * 4 : NONE, 0, 0));
  }

  keep_order();

  // ---- the wave's row: update, norm, rounded copy to LDS
  if (mine) {
    float s[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      y[j] = make_float4(__uint_as_float(yb[j].x << 16), __uint_as_float(yb[j].x & 0xffff0000u), __uint_as_float(yb[j].y << 16), __uint_as_float(yb[j].y & 0xffff0000u));
      if (a.bias) { y[j].x += bi[j].x; y[j].y += bi[j].y; y[j].z += bi[j].z; y[j].w += bi[j].w; }
      if (4 * (64 * j + lane) >= K) y[j] = v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
      s[j] = squares(y[j]);
    }
    const float ry = 1.f / sqrtf(row_sum(s) / (float)K + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j].x += y[j].x * ry * wp[j].x; v[j].y += y[j].y * ry * wp[j].y; v[j].z += y[j].z * ry * wp[j].z; v[j].w += y[j].w * ry * wp[j].w;
      s[j] = squares(v[j]);
    }
    const float rx = 1.f / sqrtf(row_sum(s) / (float)K + a.eps);
    const bool leave = wave % gridDim.x == blockIdx.x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * (64 * j + lane);
      if (c < K) {
        if (leave) *reinterpret_cast<float4*>(a.x2 + (long)wave * K + c) = v[j];
        *reinterpret_cast<uint2*>(rows + wave * PITCH + c) = make_uint2(f2bf2(v[j].x * rx * wn[j].x, v[j].y * rx * wn[j].y),
                                                                        f2bf2(v[j].z * rx * wn[j].z, v[j].w * rx * wn[j].w));
      }
    }
  }
  __syncthreads();

  // ---- product (rows past M are whatever LDS holds: only their own results are made of them)
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (wk0 + 32 * u < wk1) {
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(rows + r16 * PITCH + wk0 + 32 * u + 8 * g);
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w[u][n], acc[n], 0, 0, 0);
    }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][(4 * g + r) * LD + 16 * n + r16] = acc[n][r];
  __syncthreads();
  if (!item) return;
  auto sum = [&](int c) {
    f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll GLU ? 2 : 4
    for (int gr = 0; gr < WV / 4; ++gr) {
      auto at = [&](int i) { return *reinterpret_cast<const f32x4*>(&part[4 * gr + i][m * LD + c]); };
      t += (at(0) + at(2)) + (at(1) + at(3));
    }
    return t;
  };
  uint2 o;
  if constexpr (GLU) {      // the product's rounding, then glu_act's steps (seqmix.hip) on it
    if (2 * gc >= N) return;
    const f32x4 x1 = sum(q / 2 * 16 + 4 * (q & 1)), x2 = sum(q / 2 * 16 + 8 + 4 * (q & 1));
    float r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float gv = bf2f(f2bf(x1[j])) + bg[j], uv = bf2f(f2bf(x2[j])) + bu[j], al = 1.f;
      if (a.mode == 1) {
        gv = fminf(gv, a.limit);
        uv = fminf(fmaxf(uv, -a.limit), a.limit) + 1.f;
        al = a.alpha;
      } else if (a.mode == 2) {
        al = 1.5957691216057308f * (1.f + 0.044715f * gv * gv);
      }
      r[j] = gv * __builtin_amdgcn_rcpf(1.f + __expf(-al * gv)) * uv;
    }
    o = make_uint2(f2bf2(r[0], r[1]), f2bf2(r[2], r[3]));
    *reinterpret_cast<uint2*>(a.out + (long)m * a.ldo + gc) = o;
  } else {
    const int c = NC * tile + 4 * q;
    const f32x4 t = sum(4 * q);
    o = make_uint2(f2bf2(t[0], t[1]), f2bf2(t[2], t[3]));
    u16* d = a.out + (long)m * a.ldo + c;
    if (c + 4 <= N) *reinterpret_cast<uint2*>(d) = o;
    else
      for (int j = 0; j < 4; ++j)
        if (c + j < N) d[j] = f2bf(t[j]);
  }
}

template <bool GLU>
int launch(const TailArgs& a, int nt, hipStream_t st) {
  const dim3 grid((a.N + 16 * nt - 1) / (16 * nt));
  if (nt == 1) hipLaunchKernelGGL((tail_gemm_kernel<1, GLU>), grid, dim3(64 * WV), 0, st, a);
  else hipLaunchKernelGGL((tail_gemm_kernel<2, GLU>), grid, dim3(64 * WV), 0, st, a);
  return (int)hipGetLastError();
}
}  // namespace

// y [M, K] bf16 (rows of 8 bytes), x and x2 [M, K] f32 (not the same), W: ops.gemm.frag_weight's [ceil(N / 16)][K / 32][64][8] (GLU: paired),
// out [M, N] or [M, N / 2] (GLU), rows of 8 bytes; nt 1 or 2 tiles of 16 columns a workgroup.
extern "C" int dllm_tail_gemm(const void* y, long ldy, const float* x, float* x2, const float* w_post, const float* w_next, const float* bias,
                              float eps, const void* W, void* out, long ldo, int M, int N, int K, int nt, int glu, const float* act_bias, int mode,
                              float limit, float alpha, hipStream_t stream) {
  if (M < 1 || M > MR || K < 32 || K > MAX_K || K % 32 || N < 1 || nt < 1 || nt > 2 || x == x2 || ldy % 4 || ldo % 4) return -1;
  if (glu && (N % 16 || mode < 0 || mode > 2)) return -2;
  const TailArgs a{(const u16*)y, ldy, x, w_post, w_next, bias, x2, eps, (const u16*)W, (u16*)out, ldo, M, N, K, act_bias, mode, limit, alpha};
  return glu ? launch<true>(a, nt, stream) : launch<false>(a, nt, stream);
}
