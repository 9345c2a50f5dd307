// Chunk-parallel form of the recurrences with a scalar decay per head and token, for prompt portions
// (gfx950, wave64):
//
//     S_t = a_t S_(t-1) + b_t k_t v_t^T,    y_t = S_t^T q_t          (S: [d x dv] f32 per sequence and head)
//
//   retention / lightning   a = the head's decay, b = 1; q and k rotated (k scaled) or q, k and v SiLU'd
//   ssd                     Mamba-2: dt = softplus(logit + bias), a = exp(neg_a dt), b = dt, k = B and q = C of the
//                           head's group, v = x;  y += D x
//
// With chunks of 64 tokens, A_t the product of a over the chunk up to t and S the state before the chunk:
//
//     U   = sum_s (A_end / A_s) b_s k_s v_s^T                        chunk_sum: every chunk, head at once
//     S  <- A_end S + U                                              chunk_carry: elementwise, in chunk order
//     y_t = sum_(s <= t) (A_t / A_s) b_s (q_t . k_s) v_s + A_t S^T q_t      chunk_out: every chunk, head at once
//
// so the only serial part is one multiply-add per state entry and chunk, and a long prompt of one sequence fills the
// chip.  Everything stays in f32: products on v_mfma_f32_16x16x4_f32 (the vector ALU's rate, but its operands come
// from LDS once per 16x16 tile instead of once per row), the decay of Mamba-2 as differences of f64 sums of logarithms.
//
// MFMA layout: with lr = lane & 15, g4 = lane >> 4, A holds row lr and B column lr of contraction index g4; the
// accumulator holds rows 4 g4 .. 4 g4 + 3 of column lr.  Four products in a row take the contraction indices
// 16 blk + 4 g4 + j (j = 0 .. 3) in both operands, so a lane reads 16 bytes of a row-major row for all four; and the
// accumulator of k . q^T (rows = keys) is, register by register, the A operand of the product with v.  LDS rows are
// padded by 4 floats: 16-byte reads over 16 rows and 4-byte reads over 4 rows x 16 columns both spread over all banks.
//
// Rows go to LDS in two steps, several loads a thread in flight before the first conversion (one at a time the
// staging took half of either kernel).
//
// What bounds it: 16 heads of 128 x 128 over 6 x 1400 tokens are 12 GFLOP of f32 MFMA a layer (80 us at 157 TFLOP/s) and
// 0.5 GB of chunk states (100 us at 5.2 TB/s); chunks of 128 would halve the states and need twice the LDS.  Measured
// there (bf16 rows): sums 119, carry 53, outputs 179 us with SiLU on every row (expf and a division: 8 % of a layer).  One
// prompt of 4096 tokens, with its norm and gate: retention with 8 heads of 64 x 128 about 80 us against 1900 us
// for chunks in order (seqmix.hip); Mamba-2 with 32 heads of 128 x 64 about 150 us against 1390 us token by token
// (outer_scan.hip).
#include "chunks.h"
#include "common.h"

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }

constexpr int CS_L = 64;      // tokens per chunk
constexpr int CS_VC = 128;    // value columns per workgroup, at most
constexpr long CS_SCRATCH = 1L << 26;      // entries of chunk states (256 MB) up to which all heads go at once; else some at a time:
                                           // 16 heads of 128 x 128 from 16000 tokens on, where one head's chunks fill the chip

struct ScanArgs {
  const void *q, *k, *v;      // column 0 of the first head's q / k / v rows
  long ld, ldv;               // row strides of q and k, of v
  int kdiv;                   // heads per q / k head
  int H, d, dv, S;
  int h0, HC;                 // first head of the launch, heads that the scratch holds
  // retention / lightning
  const float *cos_sin, *decay;
  int tab_w, rot, act;
  float kscale;
  // ssd: step logits at gates[token, head]
  const void* gates;
  long ld_g;
  const float *dt_bias, *neg_a, *D;
  const int *qstart, *qlen, *ctx, *rows;
  float *state, *chunks, *ends, *out;      // state slots; [chunks][HC][d][dv], [chunks][HC] A_end (ssd); out [T, H, dv]
  int nchunks;
  int vec, rotvec;            // rows, head offsets and widths allow four elements at a time; so do rotation and its table
};

__device__ __forceinline__ float silu_f(float x) { return x / (1.f + expf(-x)); }

// four elements of a row as they lie in memory
template <typename T> struct Quad;
template <> struct Quad<u16> {
  uint2 u;
  __device__ __forceinline__ void ld(const u16* p) { u = *reinterpret_cast<const uint2*>(p); }
  __device__ __forceinline__ float4 f() const {
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xffff0000u));
  }
};
template <> struct Quad<float> {
  float4 u;
  __device__ __forceinline__ void ld(const float* p) { u = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ float4 f() const { return u; }
};
__device__ __forceinline__ float4 scale4(float4 x, float w) { return make_float4(x.x * w, x.y * w, x.z * w, x.w * w); }
__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ float4 silu4(float4 x) { return make_float4(silu_f(x.x), silu_f(x.y), silu_f(x.z), silu_f(x.w)); }

// four elements from column i of a row of n, any alignment (zeros behind the row)
template <typename T> __device__ __forceinline__ float4 ld4(const T* r, int i, int n) {
  return make_float4(i < n ? ldf(r + i) : 0.f, i + 1 < n ? ldf(r + i + 1) : 0.f, i + 2 < n ? ldf(r + i + 2) : 0.f,
                     i + 3 < n ? ldf(r + i + 3) : 0.f);
}

// four elements of a q / k row, rotated (pairs (i, i + rot / 2)) or SiLU'd: in two steps, so that a thread has the loads
// of several in flight, or at once for any alignment.  Columns from d on are zeros.
template <typename T> struct QK {
  Quad<T> x, p;
  float4 c, s;
  __device__ __forceinline__ void ld(const ScanArgs& a, const T* r, int i, int pos) {
    const int ic = min(i, a.d - 4);
    x.ld(r + ic);
    if (a.rot) {
      const int half = a.rot >> 1, f = ic < a.rot ? (ic < half ? ic : ic - half) : 0;
      p.ld(r + (ic < a.rot ? (ic < half ? ic + half : ic - half) : ic));
      const float* cs = a.cos_sin + (long)pos * a.tab_w + f;
      c = *reinterpret_cast<const float4*>(cs);
      s = *reinterpret_cast<const float4*>(cs + half);
    }
  }
  __device__ __forceinline__ float4 get(const ScanArgs& a, int i) const {
    float4 v = x.f();
    if (a.rot && i < a.rot) {
      const float4 q = p.f();
      const float g = i < (a.rot >> 1) ? -1.f : 1.f;
      v = make_float4(v.x * c.x + g * q.x * s.x, v.y * c.y + g * q.y * s.y, v.z * c.z + g * q.z * s.z, v.w * c.w + g * q.w * s.w);
    }
    if (a.act) v = silu4(v);
    return i < a.d ? v : zero4();
  }
};
template <typename T> __device__ __forceinline__ float4 ld_qk(const ScanArgs& a, const T* r, int i, int pos) {
  float4 x = ld4(r, i, a.d);
  if (i < a.rot) {
    float v[4] = {x.x, x.y, x.z, x.w};
    const int half = a.rot >> 1;
    const float* cs = a.cos_sin + (long)pos * a.tab_w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = i + j;
      if (e >= a.rot) continue;      // rot <= d
      const int f = e < half ? e : e - half;
      const float c = cs[f], s = cs[half + f], p = ldf(r + (e < half ? e + half : e - half));
      v[j] = e < half ? v[j] * c - p * s : v[j] * c + p * s;
    }
    x = make_float4(v[0], v[1], v[2], v[3]);
  }
  return a.act ? silu4(x) : x;
}

// the chunk's keys [L][KD + 4], times kscale and, with wt, a weight per token; rows past nt are zeros
template <typename T, int KD>
__device__ __forceinline__ void stage_keys(const ScanArgs& a, float* Ks, const T* kp, int nt, int p0, const float* wt) {
  constexpr int IT = CS_L * KD / 1024, U = IT < 4 ? IT : 4;
  if (a.vec && (!a.rot || a.rotvec)) {
#pragma unroll
    for (int it = 0; it < IT; it += U) {
      QK<T> x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = threadIdx.x + 256 * (it + u), t = min(e / (KD / 4), nt - 1);
        x[u].ld(a, kp + t * a.ld, (e % (KD / 4)) * 4, p0 + t);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = threadIdx.x + 256 * (it + u), t = e / (KD / 4), i = (e % (KD / 4)) * 4;
        const float w = t < nt ? (wt ? wt[t] : 1.f) * a.kscale : 0.f;
        *reinterpret_cast<float4*>(Ks + t * (KD + 4) + i) = t < nt ? scale4(x[u].get(a, i), w) : zero4();
      }
    }
  } else {
    for (int e = threadIdx.x; e < CS_L * KD / 4; e += 256) {
      const int t = e / (KD / 4), i = (e % (KD / 4)) * 4;
      *reinterpret_cast<float4*>(Ks + t * (KD + 4) + i) =
          t < nt ? scale4(ld_qk(a, kp + t * a.ld, i, p0 + t), (wt ? wt[t] : 1.f) * a.kscale) : zero4();
    }
  }
}

// Four of a token's values, rid of infinities and NaN; seen (one entry a token): 1, or NaN where the row had any.  The 4 NV threads of
// a row are neighbours in a wave.
template <int NV> __device__ __forceinline__ float4 finite4(float4 v, float* seen) {
  constexpr unsigned long long row = (1ull << (4 * NV)) - 1;
  const int lane = threadIdx.x & 63;
  const unsigned long long bad = __ballot(!(fmaf(v.y, 0.f, v.x * 0.f) + fmaf(v.w, 0.f, v.z * 0.f) == 0.f));
  if (lane % (4 * NV) == 0) *seen = (bad >> lane) & row ? __builtin_nanf("") : 1.f;
  if (bad)
    v = make_float4(v.x * 0.f == 0.f ? v.x : 0.f, v.y * 0.f == 0.f ? v.y : 0.f, v.z * 0.f == 0.f ? v.z : 0.f, v.w * 0.f == 0.f ? v.w : 0.f);
  return v;
}

// the chunk's values [L][16 NV + 4] from column 0 of vp, n of them in a row; rows past nt are zeros.  seen: as in finite4, or null
template <typename T, int NV>
__device__ __forceinline__ void stage_values(const ScanArgs& a, float* Vs, const T* vp, int nt, int n, float* seen) {
  constexpr int IT = CS_L * NV / 64, VS = 16 * NV + 4;
  if (a.vec) {
    Quad<T> x[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int e = threadIdx.x + 256 * it;
      x[it].ld(vp + min(e / (4 * NV), nt - 1) * a.ldv + min((e % (4 * NV)) * 4, n - 4));
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int e = threadIdx.x + 256 * it, t = e / (4 * NV), i = (e % (4 * NV)) * 4;
      float4 v = x[it].f();
      if (a.act) v = silu4(v);
      v = t < nt && i < n ? v : zero4();
      *reinterpret_cast<float4*>(Vs + t * VS + i) = seen ? finite4<NV>(v, seen + t) : v;
    }
  } else {
    for (int e = threadIdx.x; e < CS_L * NV * 4; e += 256) {
      const int t = e / (4 * NV), i = (e % (4 * NV)) * 4;
      float4 v = zero4();
      if (t < nt) v = ld4(vp + t * a.ldv, i, n);
      if (a.act) v = silu4(v);
      *reinterpret_cast<float4*>(Vs + t * VS + i) = seen ? finite4<NV>(v, seen + t) : v;
    }
  }
}

// one token's step and logarithm of decay, and the sum of logarithms over the chunk up to it (a lane per token)
template <typename T>
__device__ __forceinline__ void ssd_gates(const ScanArgs& a, int h, int tok0, int nt, float& dt, double& sum) {
  const int lane = threadIdx.x & 63;
  dt = 0.f;
  if (lane < nt) {
    const float x = ldf((const T*)a.gates + (long)(tok0 + lane) * a.ld_g + h) + a.dt_bias[h];
    dt = x > 20.f ? x : log1pf(expf(x));
  }
  sum = (double)a.neg_a[h] * (double)dt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double u = __shfl_up(sum, o);
    if (lane >= o) sum += u;
  }
}

// U of one (chunk, head, 128 value columns)
template <typename T, int KD, int NV, bool SSD>
__global__ void __launch_bounds__(256) chunk_sum_kernel(ScanArgs a) {
  constexpr int KS = KD + 4, VS = 16 * NV + 4;
  constexpr int WR = KD / 16 < 4 ? KD / 16 : 4, WC = 4 / WR;      // waves over the row and the column tiles
  constexpr int NR = KD / 16 / WR, NC = (NV + WC - 1) / WC;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float wt[CS_L];
  int s, c;
  if (!dllm::find_chunk<CS_L>(a.qlen, a.S, blockIdx.x, s, c)) return;
  const int h = a.h0 + blockIdx.y, v0 = blockIdx.z * CS_VC;
  const int n = a.qlen[s], t0 = c * CS_L, nt = min(CS_L, n - t0), tok0 = a.qstart[s] + t0, p0 = a.ctx[s] - n + t0;
  float* Ks = sm;                    // [L][KS]: keys times their weight
  float* Vs = sm + CS_L * KS;        // [L][VS]
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave == 0) {
    if constexpr (SSD) {
      float dt;
      double sum;
      ssd_gates<T>(a, h, tok0, nt, dt, sum);
      const double end = __shfl(sum, 63);
      wt[lane] = dt * expf((float)(end - sum));
      if (lane == 0 && v0 == 0) a.ends[(long)blockIdx.x * a.HC + blockIdx.y] = expf((float)end);
    } else {
      wt[lane] = lane < nt ? powf(a.decay[h], (float)(nt - 1 - lane)) : 0.f;
    }
  }
  stage_values<T, NV>(a, Vs, (const T*)a.v + (long)tok0 * a.ldv + (long)h * a.dv + v0, nt, min(a.dv - v0, CS_VC), nullptr);
  __syncthreads();
  stage_keys<T, KD>(a, Ks, (const T*)a.k + (long)tok0 * a.ld + (long)(h / a.kdiv) * a.d, nt, p0, wt);
  __syncthreads();
  const int wr = wave % WR, wc = wave / WR;
  f32x4 acc[NR][NC];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int b = 0; b < nt; b += 16) {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int t = b + 4 * g4 + x;
      float ka[NR], vb[NC];
#pragma unroll
      for (int i = 0; i < NR; ++i) ka[i] = Ks[t * KS + 16 * (wr + WR * i) + lr];
#pragma unroll
      for (int j = 0; j < NC; ++j) vb[j] = wc + WC * j < NV ? Vs[t * VS + 16 * (wc + WC * j) + lr] : 0.f;
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int j = 0; j < NC; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i], vb[j], acc[i][j], 0, 0, 0);
    }
  }
  float* u = a.chunks + ((long)blockIdx.x * a.HC + blockIdx.y) * a.d * a.dv;
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int r = 16 * (wr + WR * i) + 4 * g4 + x, col = v0 + 16 * (wc + WC * j) + lr;
        if (r < a.d && col < a.dv && wc + WC * j < NV) u[(long)r * a.dv + col] = acc[i][j][x];
      }
}

// chunk sums -> the state before every chunk, in place, and the state behind the last one into the slot
template <bool SSD, typename V>
__global__ void __launch_bounds__(256) chunk_carry_kernel(ScanArgs a) {
  constexpr int W = sizeof(V) / 4, AHEAD = 4;
  const int s = blockIdx.z, hc = blockIdx.y, h = a.h0 + hc;
  const int n = a.qlen[s];
  if (n <= 0) return;
  const int first = dllm::chunks_before<CS_L>(a.qlen, s);
  const int nc = min((n + CS_L - 1) / CS_L, a.nchunks - first);
  const long per = (long)a.d * a.dv, e = ((long)blockIdx.x * 256 + threadIdx.x) * W;
  if (e >= per) return;
  V* st = reinterpret_cast<V*>(a.state + ((long)a.rows[s] * a.H + h) * per + e);
  V* u = reinterpret_cast<V*>(a.chunks + ((long)first * a.HC + hc) * per + e);
  const long step = (long)a.HC * per / W;
  const float dec = SSD ? 0.f : a.decay[h], full = SSD ? 0.f : powf(dec, (float)CS_L);
  V S = {};
  if (a.ctx[s] - n > 0) S = *st;
  for (int c0 = 0; c0 < nc; c0 += AHEAD) {
    V x[AHEAD];
    float g[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const int c = min(c0 + j, nc - 1);
      x[j] = u[c * step];
      if constexpr (SSD) g[j] = a.ends[(long)(first + c) * a.HC + hc];
      else g[j] = (c + 1) * CS_L <= n ? full : powf(dec, (float)(n - c * CS_L));
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      if (c0 + j >= nc) break;
      u[(c0 + j) * step] = S;
      S = g[j] * S + x[j];
    }
  }
  *st = S;
}

// outputs of one (chunk, head, 128 value columns): wave w has tokens 16 w .. 16 w + 15
template <typename T, int KD, int NV, bool SSD>
__global__ void __launch_bounds__(256) chunk_out_kernel(ScanArgs a) {
  constexpr int KS = KD + 4, VS = 16 * NV + 4, NB = KD / 16;
  static_assert(KD * VS <= CS_L * (KS + VS), "the state takes the place of the keys and values");
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float wt[CS_L + 1];       // retention: powers of the decay; ssd: steps
  __shared__ double lg[CS_L];          // ssd: sums of log decays
  __shared__ float seen[CS_L];         // NaN: a value of the token is infinite or NaN.  It must not reach the tokens before it, whose
                                       // zero weights it would meet, so it reaches those behind as a weight
  int s, c;
  if (!dllm::find_chunk<CS_L>(a.qlen, a.S, blockIdx.x, s, c)) return;
  const int h = a.h0 + blockIdx.y, v0 = blockIdx.z * CS_VC;
  const int n = a.qlen[s], t0 = c * CS_L, nt = min(CS_L, n - t0), tok0 = a.qstart[s] + t0, p0 = a.ctx[s] - n + t0;
  float* Ks = sm;                      // [L][KS], then the state [KD][VS] from the start of sm
  float* Vs = sm + CS_L * KS;          // [L][VS]
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave == 0) {
    if constexpr (SSD) {
      float dt;
      double sum;
      ssd_gates<T>(a, h, tok0, nt, dt, sum);
      wt[lane] = dt;
      lg[lane] = sum;
    } else {
      wt[lane] = powf(a.decay[h], (float)lane);
      if (lane == 0) wt[CS_L] = powf(a.decay[h], (float)CS_L);
    }
  }
  const long kh = (long)tok0 * a.ld + (long)(h / a.kdiv) * a.d;
  stage_keys<T, KD>(a, Ks, (const T*)a.k + kh, nt, p0, nullptr);
  stage_values<T, NV>(a, Vs, (const T*)a.v + (long)tok0 * a.ldv + (long)h * a.dv + v0, nt, min(a.dv - v0, CS_VC), seen);
  // the wave's queries: row lr, dims 16 b + 4 g4 ..
  const int tq = 16 * wave + lr, tl = min(tq, nt - 1);
  float4 q[NB];
  {
    const T* r = (const T*)a.q + kh + tl * a.ld;
    if (a.vec && (!a.rot || a.rotvec)) {
      constexpr int U = NB < 4 ? NB : 4;
#pragma unroll
      for (int b = 0; b < NB; b += U) {
        QK<T> x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u].ld(a, r, 16 * (b + u) + 4 * g4, p0 + tl);
#pragma unroll
        for (int u = 0; u < U; ++u) q[b + u] = x[u].get(a, 16 * (b + u) + 4 * g4);
      }
    } else {
#pragma unroll
      for (int b = 0; b < NB; ++b) q[b] = ld_qk(a, r, 16 * b + 4 * g4, p0 + tl);
    }
  }
  __syncthreads();
  f32x4 acc[NV];
  const float skip = SSD ? a.D[h] : 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[j][x] = SSD ? skip * Vs[(16 * wave + 4 * g4 + x) * VS + 16 * j + lr] : 0.f;
  const double lq = SSD ? lg[tq] : 0.0;
  for (int b = 0; b <= wave; ++b) {      // keys 16 b .. 16 b + 15; later ones see none of these tokens
    if (16 * b >= nt) break;
    f32x4 p = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* kr = Ks + (16 * b + lr) * KS + 4 * g4;
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      const float4 kv = *reinterpret_cast<const float4*>(kr + 16 * x);
      p = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.x, q[x].x, p, 0, 0, 0);
      p = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.y, q[x].y, p, 0, 0, 0);
      p = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.z, q[x].z, p, 0, 0, 0);
      p = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.w, q[x].w, p, 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int k = 16 * b + 4 * g4 + x;
      float w = 0.f;
      if (k <= tq) w = (SSD ? wt[k] * expf((float)(lq - lg[k])) : wt[tq - k]) * seen[k];
      p[x] = k <= tq ? p[x] * w : 0.f;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const float* vr = Vs + (16 * b + 4 * g4 + x) * VS + lr;
#pragma unroll
      for (int j = 0; j < NV; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[x], vr[16 * j], acc[j], 0, 0, 0);
    }
  }
  if (c > 0 || p0 > 0) {      // (the same for the whole workgroup) a sequence starts from a zero state
    __syncthreads();
    const float* st = a.chunks + ((long)blockIdx.x * a.HC + blockIdx.y) * a.d * a.dv + v0;
    constexpr int IT = KD * NV / 64, U = IT < 8 ? IT : 8;
    if (a.dv % 4 == 0) {
      const int n = min(a.dv - v0, CS_VC);
#pragma unroll
      for (int it = 0; it < IT; it += U) {
        float4 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int e = tid + 256 * (it + u);
          x[u] = *reinterpret_cast<const float4*>(st + (long)min(e / (4 * NV), a.d - 1) * a.dv + min((e % (4 * NV)) * 4, n - 4));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int e = tid + 256 * (it + u), r = e / (4 * NV), i = (e % (4 * NV)) * 4;
          *reinterpret_cast<float4*>(sm + r * VS + i) = r < a.d && i < n ? x[u] : zero4();
        }
      }
    } else {
      for (int e = tid; e < KD * NV * 4; e += 256) {
        const int r = e / (4 * NV), i = (e % (4 * NV)) * 4;
        *reinterpret_cast<float4*>(sm + r * VS + i) = r < a.d ? ld4(st + (long)r * a.dv, i, a.dv - v0) : zero4();
      }
    }
    const float w = SSD ? expf((float)lq) : wt[tq + 1];
#pragma unroll
    for (int b = 0; b < NB; ++b) q[b] = scale4(q[b], w);
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float qv[4] = {q[b].x, q[b].y, q[b].z, q[b].w};
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float* sr = sm + (16 * b + 4 * g4 + x) * VS + lr;
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[x], sr[16 * j], acc[j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int t = 16 * wave + 4 * g4 + x;
    if (t >= nt) continue;
    float* o = a.out + ((long)(tok0 + t) * a.H + h) * a.dv + v0 + lr;
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (v0 + 16 * j + lr < a.dv) o[16 * j] = acc[j][x];
  }
}

template <typename T, bool SSD, int KD, int NV> void launch_tiles(ScanArgs a, hipStream_t st) {
  constexpr int lds = 4 * CS_L * (KD + 4 + 16 * NV + 4);
  static const bool set_ = [] {      // raised once: no attribute call inside a later stream capture
    (void)hipFuncSetAttribute((const void*)chunk_sum_kernel<T, KD, NV, SSD>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)hipFuncSetAttribute((const void*)chunk_out_kernel<T, KD, NV, SSD>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    return true;
  }();
  (void)set_;
  const long per = (long)a.d * a.dv;
  for (a.h0 = 0; a.h0 < a.H; a.h0 += a.HC) {      // the stream keeps one group's launches ahead of the next's writes
    const int n = a.HC < a.H - a.h0 ? a.HC : a.H - a.h0;
    const dim3 g(a.nchunks, n, (a.dv + CS_VC - 1) / CS_VC);
    hipLaunchKernelGGL((chunk_sum_kernel<T, KD, NV, SSD>), g, dim3(256), lds, st, a);
    if (per % 4 == 0 && (uintptr_t)a.state % 16 == 0 && (uintptr_t)a.chunks % 16 == 0)
      hipLaunchKernelGGL((chunk_carry_kernel<SSD, f32x4>), dim3((unsigned)((per / 4 + 255) / 256), n, a.S), dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((chunk_carry_kernel<SSD, float>), dim3((unsigned)((per + 255) / 256), n, a.S), dim3(256), 0, st, a);
    hipLaunchKernelGGL((chunk_out_kernel<T, KD, NV, SSD>), g, dim3(256), lds, st, a);
  }
}

template <typename T, bool SSD> int launch_chunks(const ScanArgs& a, hipStream_t st) {
#define CS_V(KD)                                                                                        \
  do {                                                                                                  \
    if (a.dv <= 32) launch_tiles<T, SSD, KD, 2>(a, st);                                                 \
    else if (a.dv <= 64) launch_tiles<T, SSD, KD, 4>(a, st);                                            \
    else launch_tiles<T, SSD, KD, 8>(a, st);                                                            \
  } while (0)
  if (a.d <= 32) CS_V(32); else if (a.d <= 64) CS_V(64); else CS_V(128);
#undef CS_V
  return (int)hipGetLastError();
}

template <typename T> int vec_ok(const ScanArgs& a) {
  const int bytes = 4 * sizeof(T);
  return a.d % 4 == 0 && a.dv % 4 == 0 && a.ld % 4 == 0 && a.ldv % 4 == 0 && (uintptr_t)a.q % bytes == 0 &&
         (uintptr_t)a.k % bytes == 0 && (uintptr_t)a.v % bytes == 0;
}

int heads_at_once(long nchunks, int H, int d, int dv) {
  const long n = CS_SCRATCH / (nchunks * ((long)d * dv + 1));
  return n < 1 ? 1 : n < H ? (int)n : H;
}

template <bool SSD> int run_chunks(ScanArgs& a, int f32, long T, float* scratch, hipStream_t st) {
  if (a.d < 1 || a.d > 128 || a.dv < 1 || a.S < 1 || T < 1) return -1;
  a.nchunks = (int)(T / CS_L) + a.S;
  a.HC = heads_at_once(a.nchunks, a.H, a.d, a.dv);
  a.chunks = scratch;
  a.ends = scratch + (long)a.nchunks * a.HC * a.d * a.dv;
  a.rotvec = a.rot % 8 == 0 && a.tab_w % 4 == 0 && (uintptr_t)a.cos_sin % 16 == 0;
  if (f32) {
    a.vec = vec_ok<float>(a);
    return launch_chunks<float, SSD>(a, st);
  }
  a.vec = vec_ok<u16>(a);
  return launch_chunks<u16, SSD>(a, st);
}

}  // namespace

// f32 entries of scratch for a step of T tokens and S sequences; 0: the width is not taken
extern "C" long dllm_chunk_scan_scratch(long T, int S, int H, int d, int dv) {
  if (d < 1 || d > 128 || dv < 1 || T < 1 || S < 1) return 0;
  const long nc = T / CS_L + S;
  return nc * heads_at_once(nc, H, d, dv) * ((long)d * dv + 1);
}

// qkvg [T, q | k | v | ..]: q and k rotated, k times kscale, or with act all three SiLU'd; out [T, H, dv] f32
extern "C" int dllm_retention_chunks(const void* qkvg, long ld, int f32, int H, int d, int dv, const float* cos_sin, int tab_w,
                                     int rot, const float* decay, float* state, const int* qstart, const int* qlen,
                                     const int* ctx, const int* rows, float* out, int S, long T, int act, float kscale,
                                     float* scratch, hipStream_t st) {
  if (rot < 0 || rot > d || (rot & 1) || (rot && rot > tab_w)) return -1;
  const char* p = (const char*)qkvg;
  const long it = f32 ? 4 : 2;
  ScanArgs a{};
  a.q = p, a.k = p + it * H * d, a.v = p + it * 2 * H * d;
  a.ld = a.ldv = ld, a.kdiv = 1, a.H = H, a.d = d, a.dv = dv, a.S = S;
  a.cos_sin = cos_sin, a.decay = decay, a.tab_w = tab_w, a.rot = rot, a.act = act, a.kscale = kscale;
  a.qstart = qstart, a.qlen = qlen, a.ctx = ctx, a.rows = rows, a.state = state, a.out = out;
  return run_chunks<false>(a, f32, T, scratch, st);
}

// xbc [T, ld] = x | B | C (convolved, activated), step logits at gates[:, head]
extern "C" int dllm_ssd_chunks(const void* xbc, long ld, const void* gates, long ld_g, int f32, int H, int dv, int N, int G,
                               const float* dt_bias, const float* neg_a, const float* D, float* state, const int* qstart,
                               const int* qlen, const int* ctx, const int* rows, int S, long T, float* out, float* scratch,
                               hipStream_t st) {
  const char* p = (const char*)xbc;
  const long it = f32 ? 4 : 2, inner = (long)H * dv;
  ScanArgs a{};
  a.v = p, a.k = p + it * inner, a.q = p + it * (inner + (long)G * N);
  a.ld = a.ldv = ld, a.kdiv = H / G, a.H = H, a.d = N, a.dv = dv, a.S = S, a.kscale = 1.f;
  a.gates = gates, a.ld_g = ld_g, a.dt_bias = dt_bias, a.neg_a = neg_a, a.D = D;
  a.qstart = qstart, a.qlen = qlen, a.ctx = ctx, a.rows = rows, a.state = state, a.out = out;
  return run_chunks<true>(a, f32, T, scratch, st);
}
