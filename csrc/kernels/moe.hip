// Mixture-of-experts FFN for Mixtral-style top-k routing — graph-capturable (no host sync).
//
//   moe_route   : one workgroup turns the top-k expert ids [T*k] into an expert-sorted pair list
//                 (perm) and a tile list (expert, first row, rows) of MT-row tiles; the tile count
//                 lives on the device, so a captured decode graph handles any routing.
//   moe_gemm13  : grouped GEMM over the tile list: rows gathered through perm straight from the
//                 token activations (no materialised permuted copy), gate and up columns of the
//                 expert's fused w13 in the same wave, SiLU(gate)*up in the epilogue -> act.
//   moe_gemm2   : grouped down projection act . w2_e^T, scaled by the pair's gate weight and
//                 written to the pair's own slot (token-major, [T*k, H] f32)
//   moe_combine : out[t] = sum_j y[t*k + j] in fixed order -> deterministic, no atomics.
// MFMA: v_mfma_f32_16x16x32_bf16; A = 16 gathered rows x 32 k (row lane&15, k 8(lane>>4)+j),
// B = 32 k x 16 weight rows (same pattern on the [N, K] weight), C row (lane>>4)*4+r, col lane&15.
// Tiles are MT = 32 rows (two MFMA row groups share every weight load); blocks past the device
// tile count exit immediately.  Weights stream with 4 k-steps of loads in flight per wave.
//
// moe_ffn_tg (the default on GPU): the same routing with BM-row tiles, then BOTH expert GEMMs on
// the LDS-tiled MFMA GEMM of tgemm.hip in grouped mode — global_load_lds ring, XOR-swizzled LDS,
// rows of the first GEMM gathered through perm by the staging addresses, the expert's weight
// slice picked per row tile, SwiGLU in the epilogue over gate/up rows interleaved in 16-row
// groups (models.llama.interleave_w13) — and a combine that applies the gate weights while
// summing each token's k expert rows (inverse permutation, fixed order, no atomics).
// act_mode 1 (squared-ReLU experts, no gate projection): the same with relu(.)^2 in the first epilogue and the
// second GEMM's rows kept in f32 up to the combine.  One of the k experts may be a shared one that every token
// runs with weight 1 (its pairs come from the router kernel), so it costs no launches of its own.  Routing
// and 8 + 1 experts of 1024 x 1024, top 2, replayed over 6 layers' weights: 1 token 52 -> 34 us, 24 tokens 59 -> 39,
// 300 tokens 87 -> 46, 4001 tokens 401 -> 138 us, against the 32-row kernels above (moe_ffn, which stay for widths
// that are no multiple of 64) with the shared expert's two GEMMs, activation and add as launches of their own.
#include "common.h"
#include "tgemm_args.h"

extern "C" int dllm_moe_norm_resadd(const void* y, int f32, const int* inv, const float* wts, int k, const float* w, float* x, void* xl,
                                    long T, int H, float eps, int groups, hipStream_t st);
extern "C" int dllm_moe_decode(const void* x, long ldx, int div, const int* ids, int P, int E, const void* w, int N, int K, int act,
                               int ks, void* out, long ldo, hipStream_t st);
extern "C" int dllm_tgemm(const void* args, int bm, int bn, int stages, int ks, int nw, int wk, int epi,
                          hipStream_t stream, int nl);

namespace {
constexpr int MT = 32;

__global__ void __launch_bounds__(1024) moe_route_kernel(const int* __restrict__ ids, int P, int E, int max_tiles,
                                                         int* __restrict__ perm, int* __restrict__ tile_e,
                                                         int* __restrict__ tile_r0, int* __restrict__ tile_n,
                                                         int* __restrict__ n_tiles, int mt = MT,
                                                         int* __restrict__ inv = nullptr) {
  // Pairs are placed in a stable order (pair index ascending within each expert).  A wave owns a run of pairs and counts them 64 at a
  // time: the lanes of an expert find each other by a ballot per bit of its number, and the first of them adds their count to the
  // wave's own row of LDS.  One wave turns the counts into every wave's first place per expert; then the waves place their
  // pairs, again without meeting.  (Counting by atomics and placing 1024 pairs at a time between barriers, each round behind its own
  // load: 12003 pairs of 9 experts 25 us, here 13.)
  __shared__ int cnt[64], off[64], toff[64], at[16][64], ntl;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nwv = blockDim.x >> 6;
  const int chunks = (P + 63) >> 6, per = (chunks + nwv - 1) / nwv, c0 = min(chunks, wv * per), c1 = min(chunks, c0 + per);
  const int bits = 32 - __clz(max(E - 1, 1));
  const unsigned long long below = (1ull << lane) - 1ull;
  auto same = [&](int e, bool ok) {      // the lanes with this lane's expert
    unsigned long long m = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 6; ++b)
      if (b < bits) {
        const bool one = (e >> b) & 1;
        const unsigned long long v = __ballot(one);
        m &= one ? v : ~v;
      }
    return m;
  };
  auto each = [&](auto&& f) {            // f(pair, expert, its lanes) over this wave's pairs, eight loads in flight
    for (int c = c0; c < c1; c += 8) {
      int id[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) id[u] = ids[min((c + u) * 64 + lane, P - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c + u < c1) {
          const int p = (c + u) * 64 + lane, e = min(max(id[u], 0), E - 1);
          const unsigned long long m = same(e, p < P);
          if (p < P) f(p, e, m);
        }
    }
  };
  at[wv][lane] = 0;
  each([&](int, int e, unsigned long long m) {
    if (!(m & below)) atomicAdd(&at[wv][e], __popcll(m));
  });
  __syncthreads();
  if (tid < 64) {   // first pair and first tile of every expert: lane e of one wave
    int c = 0;
    for (int v = 0; v < nwv; ++v) c += at[v][lane];
    const int nt = (c + mt - 1) / mt;
    int po = c, to = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int a = __shfl_up(po, o), b = __shfl_up(to, o);
      if (lane >= o) { po += a; to += b; }
    }
    cnt[tid] = c;
    off[tid] = po -= c;
    toff[tid] = to - nt;
    if (tid == 63) *n_tiles = ntl = min(to, max_tiles);
    for (int v = 0; v < nwv; ++v) {
      const int n = at[v][lane];
      at[v][lane] = po;
      po += n;
    }
  }
  __syncthreads();
  for (int i = tid; i < ntl; i += blockDim.x) {
    int e = 0;
    for (int x = 1; x < E; ++x) e += toff[x] <= i;      // experts without tiles share the next one's start: the last of them owns it
    const int r = (i - toff[e]) * mt;
    tile_e[i] = e;
    tile_r0[i] = off[e] + r;
    tile_n[i] = min(mt, cnt[e] - r);
  }
  each([&](int p, int e, unsigned long long m) {
    const int first = at[wv][e], pos = first + __popcll(m & below);
    __builtin_amdgcn_wave_barrier();      // every lane's read lies before the first one's write
    if (!(m & below)) at[wv][e] = first + __popcll(m);
    __builtin_amdgcn_wave_barrier();
    perm[pos] = p;
    if (inv != nullptr) inv[p] = pos;
  });
}

__device__ __forceinline__ void ld8(const u16* p, float* f) { unpack8(ld16(p), f); }
__device__ __forceinline__ void ld8(const float* p, float* f) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

// out[t] = sum_j wts[t k + j] * y[inv[t k + j]]  (y: expert outputs in expert-sorted row order)
template <typename T_>
__global__ void moe_combine_perm_kernel(const T_* __restrict__ y, const int* __restrict__ inv,
                                        const float* __restrict__ wts, int k, int H, long T, u16* __restrict__ out) {
  const long n8 = T * (H / 8);
  for (long v = blockIdx.x * (long)blockDim.x + threadIdx.x; v < n8; v += (long)gridDim.x * blockDim.x) {
    const long t = v / (H / 8);
    const int h = (int)(v % (H / 8)) * 8;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const long p = t * k + j;
      float f[8];
      ld8(y + (inv ? (long)inv[p] : p) * H + h, f);
      const float w = wts[p];
#pragma unroll
      for (int q = 0; q < 8; ++q) s[q] += w * f[q];
    }
    st16(out + t * (long)H + h, pack8(s));
  }
}

// The same sum rounded to bf16 and added to the residual stream, r = bf16(bf16(sum) + r), with the row's sums of squares per slice of
// `cw` columns (res_add_ssq of tgemm.hip, bit for bit, in the combine's launch): a wave per row and slice.
__global__ void __launch_bounds__(256) moe_combine_resadd_kernel(const u16* __restrict__ y, const int* __restrict__ inv,
                                                                 const float* __restrict__ wts, int k, int H, int T,
                                                                 u16* __restrict__ r, long ldr, float* __restrict__ ssq, long ssq_ld,
                                                                 int cw) {
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= T) return;
  u16* rr = r + (long)row * ldr;
  const int c1 = min(H, (int)(blockIdx.y + 1) * cw);
  float q = 0.f;
  for (int c = blockIdx.y * cw + lane * 8; c < c1; c += 512) {
    float v[8], s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    unpack8(ld16(rr + c), v);
    for (int j = 0; j < k; ++j) {
      const long p = (long)row * k + j;
      float f[8];
      ld8(y + (inv ? (long)inv[p] : p) * H + c, f);
      const float w = wts[p];
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] += w * f[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = bf2f(f2bf(v[e] + bf2f(f2bf(s[e]))));
      q += v[e] * v[e];
    }
    st16(rr + c, pack8(v));
  }
  q = wave_sum(q);
  if (lane == 0) ssq[(long)blockIdx.y * ssq_ld + row] = q;
}

__device__ __forceinline__ bf16x8 ld_or0(const u16* p, bool ok) {
  return __builtin_bit_cast(bf16x8, ok ? ld16(p) : make_uint4(0, 0, 0, 0));
}

// act[row, c] = silu(x_row . wg_c) * (x_row . wu_c); block = 4 waves x 16 columns, MT rows.
// ACT 1: experts without a gate projection, act = relu(x_row . w_c)^2 (w13 is then [E, I, H]).
template <int ACT>
__global__ void __launch_bounds__(256) moe_gemm13_kernel(const u16* __restrict__ x, long x_stride,
                                                         const int* __restrict__ perm, int k,
                                                         const int* __restrict__ tile_e,
                                                         const int* __restrict__ tile_r0,
                                                         const int* __restrict__ tile_n,
                                                         const int* __restrict__ n_tiles,
                                                         const u16* __restrict__ w13, u16* __restrict__ act, int I,
                                                         int H) {
  const int tile = blockIdx.x;
  if (tile >= *n_tiles) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col0 = blockIdx.y * 64 + wave * 16;
  if (col0 >= I) return;  // whole wave; the kernel has no block-level barrier
  const int e = tile_e[tile], r0 = tile_r0[tile], nrows = tile_n[tile];
  const int rl = lane & 15, kq = 8 * (lane >> 4);
  const u16* arow[2];
  bool aok[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int row = 16 * g + rl;
    aok[g] = row < nrows;
    const int pair = aok[g] ? perm[r0 + row] : 0;
    arow[g] = x + (long)(pair / k) * x_stride + kq;
  }
  const int n = col0 + rl;
  const bool nok = n < I;
  const u16* wg = w13 + ((long)e * (ACT ? 1 : 2) * I + (nok ? n : 0)) * H + kq;
  const u16* wu = ACT ? wg : wg + (long)I * H;
  f32x4 ag[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  f32x4 au[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  int kk = 0;
  for (; kk + 128 <= H; kk += 128) {
    bf16x8 a[4][2], bg[4], bu[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bg[s] = ld_or0(wg + kk + 32 * s, nok);
      if (!ACT) bu[s] = ld_or0(wu + kk + 32 * s, nok);
#pragma unroll
      for (int g = 0; g < 2; ++g) a[s][g] = ld_or0(arow[g] + kk + 32 * s, aok[g]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        ag[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][g], bg[s], ag[g], 0, 0, 0);
        if (!ACT) au[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][g], bu[s], au[g], 0, 0, 0);
      }
  }
  for (; kk < H; kk += 32) {
    const bf16x8 bgs = ld_or0(wg + kk, nok), bus = ld_or0(wu + kk, nok && !ACT);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const bf16x8 as = ld_or0(arow[g] + kk, aok[g]);
      ag[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as, bgs, ag[g], 0, 0, 0);
      if (!ACT) au[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as, bus, au[g], 0, 0, 0);
    }
  }
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * g + (lane >> 4) * 4 + r;
      if (row < nrows && nok) {
        const float gv = ag[g][r];
        const float rl = fmaxf(gv, 0.f);
        act[(long)(r0 + row) * I + n] = f2bf(ACT ? rl * rl : gv / (1.f + __expf(-gv)) * au[g][r]);
      }
    }
}

// y[pair, c] = gate_w[pair] * (act_row . w2_e[c]); block = 4 waves x 32 columns, MT rows.
__global__ void __launch_bounds__(256) moe_gemm2_kernel(const u16* __restrict__ act, const int* __restrict__ perm,
                                                        const float* __restrict__ wts,
                                                        const int* __restrict__ tile_e,
                                                        const int* __restrict__ tile_r0,
                                                        const int* __restrict__ tile_n,
                                                        const int* __restrict__ n_tiles, const u16* __restrict__ w2,
                                                        float* __restrict__ y, int I, int H) {
  const int tile = blockIdx.x;
  if (tile >= *n_tiles) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col0 = blockIdx.y * 128 + wave * 32;
  if (col0 >= H) return;
  const int e = tile_e[tile], r0 = tile_r0[tile], nrows = tile_n[tile];
  const int rl = lane & 15, kq = 8 * (lane >> 4);
  const u16* arow[2];
  bool aok[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int row = 16 * g + rl;
    aok[g] = row < nrows;
    arow[g] = act + (long)(r0 + (aok[g] ? row : 0)) * I + kq;
  }
  const u16* wb[2];
  bool nok[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int n = col0 + 16 * c + rl;
    nok[c] = n < H;
    wb[c] = w2 + ((long)e * H + (nok[c] ? n : 0)) * I + kq;
  }
  f32x4 acc[2][2] = {};
  int kk = 0;
  for (; kk + 128 <= I; kk += 128) {
    bf16x8 a[4][2], b[4][2];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        b[s][g] = ld_or0(wb[g] + kk + 32 * s, nok[g]);
        a[s][g] = ld_or0(arow[g] + kk + 32 * s, aok[g]);
      }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          acc[g][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][g], b[s][c], acc[g][c], 0, 0, 0);
  }
  for (; kk < I; kk += 32) {
    bf16x8 a[2], b[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      a[g] = ld_or0(arow[g] + kk, aok[g]);
      b[g] = ld_or0(wb[g] + kk, nok[g]);
    }
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        acc[g][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[g], b[c], acc[g][c], 0, 0, 0);
  }
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * g + (lane >> 4) * 4 + r;
      if (row >= nrows) continue;
      const int pair = perm[r0 + row];
      const float sc = wts[pair];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int n = col0 + 16 * c + rl;
        if (nok[c]) y[(long)pair * H + n] = sc * acc[g][c][r];
      }
    }
}

__global__ void moe_combine_kernel(const float* __restrict__ y, int k, int H, long T, u16* __restrict__ out) {
  const long n4 = T * (H / 4);
  for (long v = blockIdx.x * (long)blockDim.x + threadIdx.x; v < n4; v += (long)gridDim.x * blockDim.x) {
    const long t = v / (H / 4);
    const int h = (int)(v % (H / 4)) * 4;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const float4 q = *reinterpret_cast<const float4*>(y + ((t * k + j) * (long)H + h));
      s[0] += q.x; s[1] += q.y; s[2] += q.z; s[3] += q.w;
    }
    u16* o = out + t * (long)H + h;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = f2bf(s[j]);
  }
}
int route_threads(int P) { return P >= 1024 ? 1024 : (P + 63) / 64 * 64; }
}  // namespace

extern "C" int dllm_moe_max_tiles(int P, int E) { return (P + MT - 1) / MT + E; }

extern "C" int dllm_moe_ffn(const void* x, long x_stride, long T, int H, const int* ids, const float* wts, int k,
                            int E, const void* w13, const void* w2, int I, int* perm, int* tiles /*4 x max_tiles*/,
                            void* act, float* y, void* out, int act_mode, hipStream_t stream) {
  if (E < 1 || E > 64 || k < 1 || H % 32 != 0 || I % 32 != 0 || H % 4 != 0) return -1;
  if (T == 0) return 0;
  const int P = (int)(T * k);
  const int max_tiles = (P + MT - 1) / MT + E;
  int *te = tiles, *tr = tiles + max_tiles, *tn = tiles + 2 * max_tiles, *nt = tiles + 3 * max_tiles;
  hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(route_threads(P)), 0, stream, ids, P, E, max_tiles, perm, te, tr, tn, nt);
  if (act_mode)
    hipLaunchKernelGGL(moe_gemm13_kernel<1>, dim3(max_tiles, (I + 63) / 64), dim3(256), 0, stream, (const u16*)x,
                       x_stride, perm, k, te, tr, tn, nt, (const u16*)w13, (u16*)act, I, H);
  else
    hipLaunchKernelGGL(moe_gemm13_kernel<0>, dim3(max_tiles, (I + 63) / 64), dim3(256), 0, stream, (const u16*)x,
                       x_stride, perm, k, te, tr, tn, nt, (const u16*)w13, (u16*)act, I, H);
  hipLaunchKernelGGL(moe_gemm2_kernel, dim3(max_tiles, (H + 127) / 128), dim3(256), 0, stream, (const u16*)act, perm,
                     wts, te, tr, tn, nt, (const u16*)w2, y, I, H);
  long n4 = T * (H / 4);
  long g = (n4 + 255) / 256;
  if (g > 4096) g = 4096;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((int)g), dim3(256), 0, stream, y, k, H, T, (u16*)out);
  return (int)hipGetLastError();
}

// Tile-list size for BM-row tiles: every expert may leave one partial tile.
extern "C" int dllm_moe_max_tiles_bm(int P, int E, int bm) { return (P + bm - 1) / bm + E; }

// columns of a slice when a row's squares go to `slices` slots: whole 512-column wave passes (as dllm_res_add_ssq)
extern "C" int dllm_moe_slice(int H, int slices) { return ((H + slices - 1) / slices + 511) / 512 * 512; }

// plans: {bm, bn13, stages13, ks13, nw13, bn2, stages2, ks2, nw2}; act_mode 0: w13 interleaved [E, 2I, H] (16 gate
// rows, 16 up rows, ...), y bf16; 1: w13 [E, I, H], squared ReLU, y f32.  w2 [E, H, I]; scratch: perm/inv [P], tiles
// [4 * max_tiles + 1], act [P, I], y [P, H].  xs (f32 [T, H]): instead of `out`, xs += rmsnorm(sum) * nw in `groups` parts, and its
// rounded copy in xl (norm_resadd of seqmix.hip, in the combine's launch).  res (bf16 [T, H], act_mode 0): instead of `out`, added to the
// residual stream with the rows' squares in ssq [slots][ssq_ld].  w13f / w2f (P <= 256): the decode step's kernels on their
// fragment-major copies instead, few_ks waves a tile (perm, inv and tiles are then not read).
extern "C" int dllm_moe_ffn_tg(const void* x, long x_stride, long T, int H, const int* ids, const float* wts, int k,
                               int E, const void* w13, const void* w2, int I, int* perm, int* inv, int* tiles,
                               void* act, void* y, void* out, int act_mode, const int* plan, const float* nw, float* xs, void* xl,
                               float eps, int groups, void* res, long ldr, float* ssq, long ssq_ld, int slices, const void* w13f,
                               const void* w2f, int few_ks, hipStream_t stream) {
  if (E < 1 || E > 64 || k < 1 || H % 64 != 0 || I % 64 != 0 || x_stride % 8 || (res && (act_mode || ldr % 8 || !ssq || slices < 1))) return -1;
  if (T == 0) return 0;
  const int bm = plan[0], NI = act_mode ? I : 2 * I;
  const int P = (int)(T * k);
  const int max_tiles = (P + bm - 1) / bm + E;
  if (w13f) {      // a decode step on fragment-major weights: rows stay in pair order (moe_decode.hip)
    int rc = dllm_moe_decode(x, x_stride, k, ids, P, E, w13f, NI, H, act_mode ? 1 : 0, few_ks, act, I, stream);
    if (rc) return 3000 + rc;
    rc = dllm_moe_decode(act, I, 1, ids, P, E, w2f, H, I, act_mode ? 3 : 2, few_ks, y, H, stream);
    if (rc) return 4000 + rc;
    inv = nullptr;
  } else {
    int *te = tiles, *tr = tiles + max_tiles, *tn = tiles + 2 * max_tiles, *nt = tiles + 3 * max_tiles;
    hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(route_threads(P)), 0, stream, ids, P, E, max_tiles, perm, te, tr, tn, nt, bm,
                       inv);
    dllm::GemmArgs g{};
    g.A = (const uint16_t*)x; g.lda = x_stride; g.W = (const uint16_t*)w13; g.Y = (uint16_t*)act; g.ldy = I;
    g.M = max_tiles * bm; g.N = NI; g.K = H; g.kchunk = H; g.splits = 1;
    g.g_tiles = tiles; g.g_max = max_tiles; g.g_perm = perm; g.g_k = k; g.g_wstride = (long)NI * H;
    int rc = dllm_tgemm(&g, bm, plan[1], plan[2], plan[3], plan[4], 1, act_mode ? dllm::EPI_RELU2 : dllm::EPI_SWIGLU, stream, 0);
    if (rc) return 1000 + rc;
    dllm::GemmArgs d{};
    d.A = (const uint16_t*)act; d.lda = I; d.W = (const uint16_t*)w2; d.Y = (uint16_t*)y; d.ldy = H;
    d.M = max_tiles * bm; d.N = H; d.K = I; d.kchunk = I; d.splits = 1;
    d.g_tiles = tiles; d.g_max = max_tiles; d.g_perm = nullptr; d.g_k = 1; d.g_wstride = (long)H * I;
    rc = dllm_tgemm(&d, bm, plan[5], plan[6], plan[7], plan[8], 1, act_mode ? dllm::EPI_F32 : dllm::EPI_PLAIN, stream, 0);
    if (rc) return 2000 + rc;
  }
  if (res) {                                                                                               // ... the bf16 one
    const int cw = dllm_moe_slice(H, slices);
    hipLaunchKernelGGL(moe_combine_resadd_kernel, dim3((unsigned)((T + 3) / 4), (H + cw - 1) / cw), dim3(256), 0, stream, (const u16*)y, inv,
                       wts, k, H, (int)T, (u16*)res, ldr, ssq, ssq_ld, cw);
    return (int)hipGetLastError();
  }
  if (xs) return dllm_moe_norm_resadd(y, act_mode, inv, wts, k, nw, xs, xl, T, H, eps, groups, stream);   // the sum goes into the stream
  long n8 = T * (H / 8);
  long gr = (n8 + 255) / 256;
  if (gr > 4096) gr = 4096;
  if (act_mode)
    hipLaunchKernelGGL(moe_combine_perm_kernel<float>, dim3((int)gr), dim3(256), 0, stream, (const float*)y, inv, wts, k, H, T,
                       (u16*)out);
  else
    hipLaunchKernelGGL(moe_combine_perm_kernel<u16>, dim3((int)gr), dim3(256), 0, stream, (const u16*)y, inv, wts, k, H, T,
                       (u16*)out);
  return (int)hipGetLastError();
}
