// Router sentence encoder (MiniLM / BERT) kernels: bidirectional attention over a padded or packed batch
// the fused embedding sum + LayerNorm, and the projections of up to 64 rows (enc_gemm; more rows run on tgemm.hip, with
// the same bias / GELU / residual epilogues) and whole layers of up to 16 (enc_rows, attn_out; LayerNorm after each residual of more
// rows is in norm.hip), pooling in elementwise.hip.
//
// Reference parity: the reference encodes every query with sentence-transformers
// all-MiniLM-L6-v2 on the host (src/query_router_engine.py:181,571).
//
// encoder_attn: qkv [B*S, 3H] (row b*S + s; q | k | v, head h at columns h*D), lens [B] -> out [B*S, H].
//   Workgroup = (64-query slice, head, sequence), 4 waves x 16 queries.  The head's K and V^T for
//   the whole sequence are staged once in LDS (S <= 512: <= 68 KB) and shared by the 4 waves.
//   Per 32-key chunk a wave computes S^T = K . Q^T with mfma_f32_16x16x32_bf16 (keys as rows:
//   every lane then holds the scores of ONE query, so the online softmax is lane-local plus two
//   xor-shuffles) and O^T += V^T . P^T with P^T taken straight from the score registers (key
//   permutation k-slot 8g+j <-> key j < 4 ? 4g+j : 16+4g+j-4, the same trick as attention.hip).
//   Keys >= lens[b] are masked (padding tokens); K/V rows past S are zero in LDS.
//   starts != null: the rows of all sequences lie one behind the other (sequence b from row starts[b], lens[b] of them, S the
//   longest), and no row is padding: 96 texts of 6 to 70 words are 3800 rows instead of 6912, and every launch of the encoder
//   takes about that share of its time (GEMMs 606 -> 406 us, attention 101 -> 79).
#include "common.h"

namespace {
constexpr float LOG2E = 1.4426950408889634f;

template <int D>
__global__ void __launch_bounds__(256) encoder_attn_kernel(const u16* __restrict__ qkv, const int* __restrict__ lens,
                                                           u16* __restrict__ out, int Smax, int nh, float scale_log2,
                                                           const int* __restrict__ starts, int T) {
  constexpr int KSTEPS = D / 32, NT = D / 16, CPR = D / 8;  // 16-B chunks per head row
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int b = blockIdx.z, h = blockIdx.y;
  const long row0 = starts ? min(max(starts[b], 0), T) : b * (long)Smax;
  // rows of this sequence (packed) or of every one (padded); the LDS holds Smax of them
  const int S = starts ? (int)min((long)min(max(lens[b], 0), Smax), T - row0) : Smax;
  if ((int)blockIdx.x * 64 >= S) return;     // the whole workgroup
  const int SP = (S + 31) & ~31;
  const int VLD = SP + 8;  // V^T row stride (bf16): 16-B pad against bank conflicts
  u16* sk = reinterpret_cast<u16*>(smem);    // [SP][D]
  u16* sv = sk + SP * D;                     // [D][VLD]
  const int H = nh * D;
  const long ld = 3L * H;
  const u16* base = qkv + row0 * ld;
  const int len = min(lens[b], S);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, rl = lane & 15;
  const int q0 = (int)blockIdx.x * 64 + wave * 16;  // this wave's first query row
  const int q = q0 + rl;                             // this lane's query row
  bf16x8 qf[KSTEPS];                                 // on its way beside the keys: behind the barrier it was a trip of its own
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s)
    qf[s] = __builtin_bit_cast(bf16x8, q < S ? ld16(base + (long)q * ld + h * D + 8 * g + 32 * s) : make_uint4(0, 0, 0, 0));

  // ---- stage K rows and V^T for the whole sequence (zero past S)
  for (int e = threadIdx.x; e < SP * CPR; e += blockDim.x) {
    const int key = e / CPR, c = (e % CPR) * 8;
    uint4 kv = make_uint4(0, 0, 0, 0), vv = make_uint4(0, 0, 0, 0);
    if (key < S) {
      kv = ld16(base + (long)key * ld + H + h * D + c);
      vv = ld16(base + (long)key * ld + 2 * H + h * D + c);
    }
    st16(sk + key * D + c, kv);
    const uint32_t w[4] = {vv.x, vv.y, vv.z, vv.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sv[(c + 2 * j) * VLD + key] = (u16)(w[j] & 0xffffu);
      sv[(c + 2 * j + 1) * VLD + key] = (u16)(w[j] >> 16);
    }
  }
  __syncthreads();

  if (q0 >= S) return;                               // wave-uniform: no barrier follows
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  for (int kc = 0; kc < len; kc += 32) {
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      const bf16x8 k0 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(sk + (kc + rl) * D + 8 * g + 32 * s));
      const bf16x8 k1 =
          __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(sk + (kc + 16 + rl) * D + 8 * g + 32 * s));
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qf[s], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qf[s], s1, 0, 0, 0);
    }
    float p[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] = (kc + 4 * g + e < len) ? s0[e] * scale_log2 : -INFINITY;
      p[4 + e] = (kc + 16 + 4 * g + e < len) ? s1[e] * scale_log2 : -INFINITY;
    }
    float mloc = p[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mloc = fmaxf(mloc, p[j]);
    mloc = lane_max(mloc, 16);
    mloc = lane_max(mloc, 32);
    const float m_new = fmaxf(m_run, mloc);  // finite: key kc < len is always valid
    const float alpha = exp2f(m_run - m_new);
    float lsum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) { p[j] = exp2f(p[j] - m_new); lsum += p[j]; }
    lsum = lane_add(lsum, 16);
    lsum = lane_add(lsum, 32);
    l_run = l_run * alpha + lsum;
    m_run = m_new;
    const bf16x8 pf = __builtin_bit_cast(bf16x8, pack8(p));
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const u16* vr = sv + (16 * n + rl) * VLD + kc + 4 * g;
      const uint2 a0 = *reinterpret_cast<const uint2*>(vr), a1 = *reinterpret_cast<const uint2*>(vr + 16);
      const uint4 vv = make_uint4(a0.x, a0.y, a1.x, a1.y);
      acc[n] *= alpha;
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vv), pf, acc[n], 0, 0, 0);
    }
  }
  if (q >= S) return;
  // acc[n][e] = O^T[dim 16n + 4g + e][query rl]: 4 consecutive dims -> one 8-B store
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  u16* op = out + (row0 + q) * H + h * D;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const uint32_t lo = f2bf2(acc[n][0] * inv, acc[n][1] * inv);
    const uint32_t hi = f2bf2(acc[n][2] * inv, acc[n][3] * inv);
    *reinterpret_cast<uint2*>(op + 16 * n + 4 * g) = make_uint2(lo, hi);
  }
}

// ---- projections of few rows: y = x . w^T + bias, then erf-GELU, or added to y.  A workgroup takes 16 columns and all rows
// (up to 16 MT); its NW waves share K, KS steps of 32 each with every operand in flight at once, and meet in LDS.  Weights and
// rows come straight to registers (a weight is used by one workgroup, the rows are a few KB in L2).  Bound by one load's latency,
// the launch and the exchange; the LDS-tiled GEMM adds a ring's fill and, for long K, a split's exchange through memory: 16 rows,
// 384 -> 1152 / 384 -> 384 / 384 -> 1536 / 1536 -> 384 columns 2.9 / 3.5 / 3.5 / 5.4 us against 5.4 / 5.6 / 7.7 / 9.4.
enum { ENC_PLAIN = 0, ENC_RESADD = 1, ENC_QKV = 2, ENC_GELU = 4 };

// Loads of values that are used behind conditions, waited for at once: left to itself the compiler moves each to its use, and each then
// has a latency of its own (in a layer of 16 rows, us: attention and output 6.1 -> 5.2, the two products of rows 6.0 -> 4.9 and 5.3 -> 4.5, down 5.6 -> 5.4)
template <typename F>
__device__ __forceinline__ void arrived(F& f) { asm volatile("" : "+v"(f)); }

// KS k-steps of a wave at a time, so many that a wave's come out even where that can be (loads that do not exist are taken from those that do:
// 1024 -> 1024 columns on 64 rows, 16 waves of 2 steps, 9.4 us three at a time, 7.3)
template <int MT, int NW, int EPI, int KS>
__global__ void __launch_bounds__(64 * NW) enc_gemm_kernel(const u16* __restrict__ X, long ldx, const u16* __restrict__ W,
                                                           const u16* __restrict__ bias, u16* __restrict__ Y, long ldy, int M, int N,
                                                           int K) {
  constexpr int RS = 20;      // LDS rows of 16 + 4 floats reach every bank
  __shared__ __attribute__((aligned(16))) float red[NW][MT * 16][RS];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.x * 16;
  const int steps = K / 32, per = (steps + NW - 1) / NW, s0 = w * per, s1 = min(steps, s0 + per);
  const u16* wr = W + (long)(col0 + lr) * K + 8 * g;
  const u16* xr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = X + (long)min(16 * m + lr, M - 1) * ldx + 8 * g;   // rows past M repeat the last and are dropped
  const int row = threadIdx.x >> 2, c = 4 * (threadIdx.x & 3);     // this thread's outputs below: 64 rows a pass
  const u16x4 b = *reinterpret_cast<const u16x4*>(bias + col0 + c);
  u16x4 r = {};
  if (EPI == ENC_RESADD) r = *reinterpret_cast<const u16x4*>(Y + (long)min(row, M - 1) * ldy + col0 + c);
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += KS) {
    bf16x8 wf[KS], xf[KS][MT];
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const int k = 32 * min(s + u, s1 - 1);
      wf[u] = __builtin_bit_cast(bf16x8, ld16(wr + k));
#pragma unroll
      for (int m = 0; m < MT; ++m) xf[u][m] = __builtin_bit_cast(bf16x8, ld16(xr[m] + k));
    }
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      arrived(wf[u]);
#pragma unroll
      for (int m = 0; m < MT; ++m) arrived(xf[u][m]);
    }
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (s + u >= s1) break;
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[u][m], wf[u], acc[m], 0, 0, 0);
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[w][16 * m + 4 * g + i][lr] = acc[m][i];
  __syncthreads();
  if (row >= M) return;               // M <= 64 rows of four threads each: the first 256 threads
  f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][row][c]);
#pragma unroll
  for (int j = 1; j < NW; ++j) v += *reinterpret_cast<const f32x4*>(&red[j][row][c]);
  u16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float z = bf2f(f2bf(v[i] + bf2f(b.v[i])));               // the projection's own rounding, as in the tiled form
    o.v[i] = f2bf(EPI == ENC_GELU ? gelu_bf(z) : EPI == ENC_RESADD ? z + bf2f(r.v[i]) : z);
  }
  *reinterpret_cast<u16x4*>(Y + (long)row * ldy + col0 + c) = o;
}

template <int MT, int NW, int KS>
int launch_enc_gemm(const u16* x, long ldx, const u16* w, const u16* bias, u16* y, long ldy, int M, int N, int K, int epi, hipStream_t st) {
  const dim3 g(N / 16), b(64 * NW);
  if (epi == ENC_PLAIN) hipLaunchKernelGGL((enc_gemm_kernel<MT, NW, ENC_PLAIN, KS>), g, b, 0, st, x, ldx, w, bias, y, ldy, M, N, K);
  else if (epi == ENC_RESADD) hipLaunchKernelGGL((enc_gemm_kernel<MT, NW, ENC_RESADD, KS>), g, b, 0, st, x, ldx, w, bias, y, ldy, M, N, K);
  else if (epi == ENC_GELU) hipLaunchKernelGGL((enc_gemm_kernel<MT, NW, ENC_GELU, KS>), g, b, 0, st, x, ldx, w, bias, y, ldy, M, N, K);
  else return -1;
  return (int)hipGetLastError();
}

template <int MT, int NW>
int launch_enc_gemm(const u16* x, long ldx, const u16* w, const u16* bias, u16* y, long ldy, int M, int N, int K, int epi, hipStream_t st) {
  const int per = (K / 32 + NW - 1) / NW;      // k-steps a wave: 3 of 384 and 1536 columns
  if (per % 3 == 0) return launch_enc_gemm<MT, NW, 3>(x, ldx, w, bias, y, ldy, M, N, K, epi, st);
  if (per % 4 == 0) return launch_enc_gemm<MT, NW, 4>(x, ldx, w, bias, y, ldy, M, N, K, epi, st);
  if (per % 2 == 0) return launch_enc_gemm<MT, NW, 2>(x, ldx, w, bias, y, ldy, M, N, K, epi, st);
  return launch_enc_gemm<MT, NW, 3>(x, ldx, w, bias, y, ldy, M, N, K, epi, st);
}

// ---- whole layers of up to 16 rows (H <= 384) in four launches instead of seven: [LayerNorm +] QKV, attention + output + residual,
// LayerNorm + up + GELU, down + residual (enc_gemm).  A launch of this size costs 3 to 4 us whatever it does, so a workgroup
// recomputes what passed between two of them for all rows (16 rows x 384 columns are a few KB in L2) and multiplies it with its 16
// columns of the next product.  All waves share the first part, a row or a head each; what they leave in LDS as bf16 rows one wave
// multiplies, in enc_gemm's four partial sums, which makes its bits.  Six layers of 384 / 1536 on 16 rows, in a captured graph: 144 -> 124 us.  More rows
// repeat too much: with as many row tiles a workgroup, 32 rows took 185 us against 171, 64 299 against 214.
constexpr int FEW_M = 16, FEW_K = 384, FEW_LD = FEW_K + 8;      // most rows and columns; LDS rows 16 bytes apart in the banks
struct FewW {
  bf16x8 f[4][3];
  __device__ __forceinline__ void load(const u16* __restrict__ wr, int steps) {
    const int per = (steps + 3) / 4;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < 3; ++u) f[j][u] = __builtin_bit_cast(bf16x8, ld16(wr + 32 * min(j * per + min(u, per - 1), steps - 1)));
  }
  __device__ __forceinline__ f32x4 mul(const u16* a, int steps) const {     // a: this lane's row and columns in LDS
    const int per = (steps + 3) / 4;
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      bf16x8 x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(a + 32 * min(j * per + u, steps - 1)));
#pragma unroll
      for (int j = 0; j < 4; ++j) arrived(x[j]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (u < per && j * per + u < steps) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j], f[j][u], acc[j], 0, 0, 0);
    }
    return ((acc[0] + acc[1]) + acc[2]) + acc[3];
  }
};

// What a row is made of where the embeddings are summed in the launch (embed_ln_kernel's arithmetic)
struct FewEmb { const int *ids, *at; const u16 *word, *pos, *type0; int S, vocab; };

// EPI ENC_QKV: columns of q and k as they are, to Y; those of v transposed, to Vt [H][16], zero from row M on, as attn_out reads them.
// ENC_GELU as in enc_gemm.  IN 1: X is the sum that a LayerNorm takes (norm.hip's arithmetic, a wave a row); 2: that sum is made here, of
// the embeddings `e` (6.2 us for 4.6: the ids come first; as a launch of its own 4 and the gap between two); the first workgroup stores its rows to Xn for the residual sum that follows.
template <int EPI, int IN>
__global__ void __launch_bounds__(1024) enc_rows_kernel(const u16* __restrict__ X, const u16* __restrict__ W, const u16* __restrict__ bias,
                                                        u16* __restrict__ Y, int M, int N, int K, const u16* __restrict__ lnw,
                                                        const u16* __restrict__ lnb, float eps, u16* __restrict__ Xn, u16* __restrict__ Vt,
                                                        FewEmb e) {
  constexpr bool LN = IN != 0;
  __shared__ __attribute__((aligned(16))) u16 sx[FEW_M * FEW_LD];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.x * 16, steps = K / 32, c = 8 * lane;
  uint4 xv = {}, gw = {}, gb = {}, pv = {}, tv = {};
  FewW wf;
  float b = 0.f;
  const int t = min(w, M - 1);        // rows past M repeat the last and are dropped
  const u16 *xr = X + (long)t * K, *pr = nullptr;
  if constexpr (IN == 2) {
    xr = e.word + (long)min(max(e.ids[t], 0), e.vocab - 1) * K;
    pr = e.pos + (long)min(max(e.at[t], 0), e.S - 1) * K;
  }
  if (c < K) {
    xv = ld16(xr + c);
    if constexpr (IN == 2) { pv = ld16(pr + c); tv = ld16(e.type0 + c); }
    if (LN) { gw = ld16(lnw + c); gb = ld16(lnb + c); }
  }
  if (w == 0) {
    wf.load(W + (long)(col0 + lr) * K + 8 * g, steps);
    b = bf2f(bias[col0 + lr]);
  }
  if (LN) {
    float v[8], s = 0.f, q = 0.f, ga[8], be[8];
    unpack8(xv, v);
    if constexpr (IN == 2) {
      float a[8], y[8];
      unpack8(pv, a);
      unpack8(tv, y);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = v[j] + a[j] + y[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) s += v[j];
    const float mean = wave_sum(s) / K;
    if (c < K)
#pragma unroll
      for (int j = 0; j < 8; ++j) { const float d = v[j] - mean; q += d * d; }
    const float rstd = rsqrtf(wave_sum(q) / K + eps);
    unpack8(gw, ga);
    unpack8(gb, be);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (v[j] - mean) * rstd * ga[j] + be[j];
    xv = pack8(v);
    if (blockIdx.x == 0 && w < M && c < K) st16(Xn + (long)w * K + c, xv);
  }
  if (c < K) st16(sx + w * FEW_LD + c, xv);
  __syncthreads();
  if (w > 0) return;
  const f32x4 v = wf.mul(sx + lr * FEW_LD + 8 * g, steps);       // column lr of rows 4g..4g + 3
  if (EPI == ENC_QKV && 3 * col0 >= 2 * N) {          // N = 3 H, and H in whole tiles of 16
    u16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = 4 * g + i < M ? f2bf(v[i] + b) : 0;
    *reinterpret_cast<u16x4*>(Vt + (long)(col0 - N / 3 * 2 + lr) * FEW_M + 4 * g) = o;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * g + i < M) {
      const float z = bf2f(f2bf(v[i] + b));
      Y[(long)(4 * g + i) * N + col0 + lr] = f2bf(EPI == ENC_GELU ? gelu_bf(z) : z);
    }
}

// y += attention(qkv) . w^T + bias.  A wave takes a head, all queries and keys.  S^T = K . Q^T leaves a query's scores in one lane
// column and P^T feeds O^T = V^T . P^T as in encoder_attn, in its key order (keys 16 to 31 of a step are zero).  Rows of other texts
// are masked by the text's bounds; where a head's values are not all finite (0 times one is NaN) each text is multiplied by itself.
template <int D>
__global__ void __launch_bounds__(64 * FEW_K / D) attn_out_kernel(const u16* __restrict__ qkv, const u16* __restrict__ Vt,
                                                                  const u16* __restrict__ W, const u16* __restrict__ bias,
                                                                  u16* __restrict__ Y, int M, int nh, float scale_log2,
                                                                  const int* __restrict__ starts, const int* __restrict__ lens, int B,
                                                                  int Smax) {
  constexpr int KST = D / 32, NT = D / 16;
  __shared__ __attribute__((aligned(16))) u16 so[FEW_M * FEW_LD];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.x * 16, H = nh * D, steps = H / 32;
  const u16* qp = qkv + (long)min(lr, M - 1) * (3 * H) + w * D + 8 * g;
  bf16x8 qf[KST], kf[KST], vf[NT];
#pragma unroll
  for (int u = 0; u < KST; ++u) {
    qf[u] = __builtin_bit_cast(bf16x8, ld16(qp + 32 * u));
    kf[u] = __builtin_bit_cast(bf16x8, ld16(qp + H + 32 * u));
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const uint2 x = *reinterpret_cast<const uint2*>(Vt + (long)(w * D + 16 * n + lr) * FEW_M + 4 * g);
    vf[n] = __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, 0, 0));
  }
  int ts = starts[min(lane, B - 1)], tn = lens[min(lane, B - 1)];
  FewW wf;
  float b = 0.f, r[4] = {};
  if (w == 0) {
    wf.load(W + (long)(col0 + lr) * H + 8 * g, steps);
    b = bf2f(bias[col0 + lr]);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = bf2f(Y[(long)min(4 * g + i, M - 1) * H + col0 + lr]);
  }
  arrived(ts);
  arrived(tn);
  ts = lane < B ? min(max(ts, 0), M) : 0;      // text `lane`: first row, rows
  tn = lane < B ? min(min(max(tn, 0), Smax), M - ts) : 0;
  int q0 = 0, q1 = 0;                  // the keys of this lane's query
  for (int t = 0; t < B; ++t) {
    const int a = __builtin_amdgcn_readlane(ts, t), e = a + __builtin_amdgcn_readlane(tn, t);
    if (lr >= a && lr < e) q0 = a, q1 = e;
  }
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < KST; ++u) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u], qf[u], s, 0, 0, 0);
  float p[8] = {}, mx = -INFINITY, l = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    p[i] = 4 * g + i >= q0 && 4 * g + i < q1 ? s[i] * scale_log2 : -INFINITY;
    mx = fmaxf(mx, p[i]);
  }
  mx = lane_max(mx, 16);
  mx = lane_max(mx, 32);
  if (mx == -INFINITY) mx = 0.f;       // a row of no text (or past M): every weight 0
#pragma unroll
  for (int i = 0; i < 4; ++i) { p[i] = exp2f(p[i] - mx); l += p[i]; }
  l = lane_add(l, 16);
  l = lane_add(l, 32);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const bf16x8 pf = __builtin_bit_cast(bf16x8, pack8(p));
  bool lost = false;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const uint4 x = __builtin_bit_cast(uint4, vf[n]);
    const unsigned e = 0x7f80u;      // an exponent of ones: an infinity or NaN
    lost |= (x.x & e) == e || (x.x >> 16 & e) == e || (x.y & e) == e || (x.y >> 16 & e) == e;
  }
  const bool apart = __any(lost);
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    if (!apart) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[n], pf, o, 0, 0, 0);
    else
      for (int t = 0; t < B; ++t) {
        const int a = __builtin_amdgcn_readlane(ts, t), e = a + __builtin_amdgcn_readlane(tn, t), k = 4 * g;
        uint4 v = __builtin_bit_cast(uint4, vf[n]);
        v.x &= (k >= a && k < e ? 0xffffu : 0u) | (k + 1 >= a && k + 1 < e ? 0xffff0000u : 0u);
        v.y &= (k + 2 >= a && k + 2 < e ? 0xffffu : 0u) | (k + 3 >= a && k + 3 < e ? 0xffff0000u : 0u);
        const f32x4 mine = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v), pf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        if (lr >= a && lr < e) o = mine;
      }
    u16x4 z;
#pragma unroll
    for (int i = 0; i < 4; ++i) z.v[i] = f2bf(o[i] * inv);
    *reinterpret_cast<u16x4*>(so + lr * FEW_LD + w * D + 16 * n + 4 * g) = z;
  }
  __syncthreads();
  if (w > 0) return;
  const f32x4 v = wf.mul(so + lr * FEW_LD + 8 * g, steps);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * g + i < M) Y[(long)(4 * g + i) * H + col0 + lr] = f2bf(bf2f(f2bf(v[i] + b)) + r[i]);
}

// out[t] = LayerNorm(word[ids[t]] + pos[p] + type0) * w + b, p = at[t] or t % S   (one wave per token, H <= 2048)
__global__ void __launch_bounds__(256) embed_ln_kernel(const int* __restrict__ ids, const u16* __restrict__ word,
                                                       const u16* __restrict__ pos, const u16* __restrict__ type0,
                                                       const u16* __restrict__ w, const u16* __restrict__ bias,
                                                       u16* __restrict__ out, int T, int S, int H, int vocab, float eps,
                                                       const int* __restrict__ at) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  const int id = min(max(ids[t], 0), vocab - 1);
  const u16* wr = word + (long)id * H;
  const u16* pr = pos + (long)(at ? min(max(at[t], 0), S - 1) : t % S) * H;
  float x[4][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = (lane + 64 * i) * 8;
    if (c < H) {
      float a[8], p[8], y[8];
      unpack8(ld16(wr + c), a);
      unpack8(ld16(pr + c), p);
      unpack8(ld16(type0 + c), y);
#pragma unroll
      for (int j = 0; j < 8; ++j) { x[i][j] = a[j] + p[j] + y[j]; s += x[i][j]; }
    }
  }
  const float mean = wave_sum(s) / H;
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if ((lane + 64 * i) * 8 < H)
#pragma unroll
      for (int j = 0; j < 8; ++j) { const float d = x[i][j] - mean; v += d * d; }
  const float rstd = rsqrtf(wave_sum(v) / H + eps);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = (lane + 64 * i) * 8;
    if (c < H) {
      float gw[8], gb[8], y[8];
      unpack8(ld16(w + c), gw);
      unpack8(ld16(bias + c), gb);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = (x[i][j] - mean) * rstd * gw[j] + gb[j];
      st16(out + (long)t * H + c, pack8(y));
    }
  }
}
}  // namespace

extern "C" int dllm_encoder_attention(const void* qkv, const int* lens, void* out, int B, int S, int nh, int d,
                                      float scale, const int* starts, int T, hipStream_t stream) {
  if (B <= 0 || S <= 0) return 0;
  if (S > 512) return -1;
  const int SP = (S + 31) / 32 * 32;
  const size_t lds = (size_t)SP * d * 2 + (size_t)d * (SP + 8) * 2;
  const dim3 grid((S + 63) / 64, nh, B);
  static const int attr_rc = [] {  // allow > 64 KB of dynamic LDS (S up to 512)
    int rc = (int)hipFuncSetAttribute((const void*)encoder_attn_kernel<32>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    rc |= (int)hipFuncSetAttribute((const void*)encoder_attn_kernel<64>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return rc;
  }();
  if (attr_rc != 0 && lds > 64 * 1024) return -3;
  switch (d) {
    case 32:
      hipLaunchKernelGGL(encoder_attn_kernel<32>, grid, dim3(256), lds, stream, (const u16*)qkv, lens, (u16*)out, S, nh,
                         scale * LOG2E, starts, T);
      break;
    case 64:
      hipLaunchKernelGGL(encoder_attn_kernel<64>, grid, dim3(256), lds, stream, (const u16*)qkv, lens, (u16*)out, S, nh,
                         scale * LOG2E, starts, T);
      break;
    default:
      return -2;
  }
  return (int)hipGetLastError();
}

extern "C" int dllm_embed_ln(const int* ids, const void* word, const void* pos, const void* type0, const void* w,
                             const void* b, void* out, int T, int S, int H, int vocab, float eps, const int* at,
                             hipStream_t stream) {
  if (H % 8 || H > 2048) return -1;
  if (T <= 0) return 0;
  hipLaunchKernelGGL(embed_ln_kernel, dim3((T + 3) / 4), dim3(256), 0, stream, ids, (const u16*)word, (const u16*)pos,
                     (const u16*)type0, (const u16*)w, (const u16*)b, (u16*)out, T, S, H, vocab, eps, at);
  return (int)hipGetLastError();
}

// May enc_gemm take it?  Up to 64 rows, where it still wins on every shape (64 rows: 4.1 / 4.8 / 4.8 / 9.5 us against 5.5 / 6.2 / 7.7 / 10.2);
// past that a workgroup re-reads more rows than its weights.
extern "C" int dllm_enc_gemm_ok(int M, int N, int K) { return M >= 1 && M <= 64 && N % 16 == 0 && K % 32 == 0; }

// y [M, N] = x [M, K] . w [N, K]^T + bias; epi 0 plain, 1 added to y, 4 erf-GELU.  Rows, weights and bias 16-byte aligned
extern "C" int dllm_enc_gemm(const void* x, long ldx, const void* w, const void* bias, void* y, long ldy, int M, int N, int K, int epi,
                             hipStream_t st) {
  if (!dllm_enc_gemm_ok(M, N, K) || ldx % 8 || ldy % 4 || (((uintptr_t)x | (uintptr_t)w) & 15) || (((uintptr_t)y | (uintptr_t)bias) & 7)) return -1;
#define ENCG(MT)                                                                                                                     \
  return K <= 768 ? launch_enc_gemm<MT, 4>((const u16*)x, ldx, (const u16*)w, (const u16*)bias, (u16*)y, ldy, M, N, K, epi, st)       \
                  : launch_enc_gemm<MT, 16>((const u16*)x, ldx, (const u16*)w, (const u16*)bias, (u16*)y, ldy, M, N, K, epi, st)
  if (M <= 16) ENCG(1);
  if (M <= 32) ENCG(2);
  if (M <= 48) ENCG(3);
  ENCG(4);
#undef ENCG
}

// May a whole layer take dllm_enc_few_layer?  (16 rows: above at enc_rows)
extern "C" int dllm_enc_few_ok(int M, int nh, int d, int I, int B) {
  return M >= 1 && M <= FEW_M && B >= 1 && B <= 64 && (d == 32 || d == 64) && nh >= 1 && nh * d <= FEW_K && I >= 32 && I % 32 == 0;
}

// One layer on M packed rows.  x [M, H]: the rows, or (ln0w) where they go: they are the LayerNorm of the sums in y, or with ids of the sums of
// embeddings word[ids] + pos[at] + type0.  Leaves the next sums in y.  w: QKV w, b, output w, b, norm w, b, up w, b, down w, b.  qkv [M, 3H], vt [H, 16],
// f [M, I].  Operands 16-byte aligned, rows contiguous.
extern "C" int dllm_enc_few_layer(void* x, void* y, void* qkv, void* vt, void* f, const void* const* w, const void* ln0w, const void* ln0b,
                                  int M, int nh, int d, int I, float eps, float scale, const int* starts, const int* lens, int B, int S,
                                  const int* ids, const int* at, const void* word, const void* pos, const void* type0, int vocab, hipStream_t st) {
  if (!dllm_enc_few_ok(M, nh, d, I, B) || (ids && !ln0w)) return -1;
  u16 *X = (u16*)x, *Y = (u16*)y, *Q = (u16*)qkv, *V = (u16*)vt, *F = (u16*)f;
  const u16* const* W = reinterpret_cast<const u16* const*>(w);
  const int H = nh * d;
  const dim3 rows(64 * FEW_M), heads(64 * nh);
  const FewEmb e{ids, at, (const u16*)word, (const u16*)pos, (const u16*)type0, S, vocab};
#define QKV(IN, FROM) \
  hipLaunchKernelGGL((enc_rows_kernel<ENC_QKV, IN>), dim3(3 * H / 16), rows, 0, st, FROM, W[0], W[1], Q, M, 3 * H, H, (const u16*)ln0w, (const u16*)ln0b, eps, X, V, e)
  if (ids) QKV(2, X); else if (ln0w) QKV(1, Y); else QKV(0, X);
#undef QKV
  if (d == 32) hipLaunchKernelGGL(attn_out_kernel<32>, dim3(H / 16), heads, 0, st, Q, V, W[2], W[3], X, M, nh, scale * LOG2E, starts, lens, B, S);
  else hipLaunchKernelGGL(attn_out_kernel<64>, dim3(H / 16), heads, 0, st, Q, V, W[2], W[3], X, M, nh, scale * LOG2E, starts, lens, B, S);
  hipLaunchKernelGGL((enc_rows_kernel<ENC_GELU, 1>), dim3(I / 16), rows, 0, st, X, W[6], W[7], F, M, I, H, W[4], W[5], eps, Y, nullptr, e);
  const int rc = (int)hipGetLastError();
  return rc ? rc : dllm_enc_gemm(F, I, W[8], W[9], Y, H, M, H, I, ENC_RESADD, st);
}
