// Gated delta rule (gfx950, wave64).
//
// Per head, with unit vectors q (times dim^-1/2) and k, a decay g in (0, 1) and a write strength
// beta in (0, 1) per token:
//     S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
// Every value column j of S is an independent recurrence over its own [dim] vector:
//     a = S_j . k,  b = S_j . q   (both on the state before the token)
//     u_j = beta (v_j - g a);   o_j = g b + u_j (k . q);   S_j <- g S_j + k u_j
// so the kernel gives a column to 16 lanes (a DPP row: the two dot products are row rotations), a
// workgroup 16 columns of one (sequence, head), and walks the tokens in order.  Tokens are staged in
// groups of 16: raw q / k rows in LDS, unit norms and k . q by one DPP row per token, beta and the decay
// (sigmoid, softplus, two exponentials) by one lane per token, so the serial part of a token is two
// multiply-add sweeps over the lane's state registers and the row sums.  A group's inputs are fetched
// into registers while the previous group's recurrence runs.  All of it is f32; the
// state [slots, heads, vdim, dim] keeps a column contiguous.  Prompt portions take 16 tokens at a time
// (delta_prep, delta_tile).  delta_finish norms each head's output
// (unit RMS times a weight shared by the heads) and applies the SiLU gate.
#include "common.h"
#include "chunks.h"

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <typename T> __device__ __forceinline__ void stf(T* p, float v);
template <> __device__ __forceinline__ void stf<u16>(u16* p, float v) { *p = f2bf(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }

__device__ __forceinline__ float row16_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));  // row_ror:8
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));  // row_ror:4
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false));  // row_ror:2
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false));  // row_ror:1
  return v;
}

constexpr int DR_TT = 16;   // tokens per staged group
constexpr int DR_COLS = 16; // value columns per workgroup

// NS: state entries per lane; lane `sub` of a column owns dims sub * NS .. sub * NS + NS - 1, kept in
// LDS at [r * 16 + sub] so that the 16 lanes of a row read consecutive words.
// VL (bf16, rows of whole 16-byte vectors): q / k rows are fetched as 16-byte vectors, 8 dims a thread,
// instead of NS scattered 2-byte loads a thread.
template <typename T, int NS, bool VL>
__global__ void __launch_bounds__(256) delta_rule_kernel(const T* __restrict__ qkv, long ldq, const T* __restrict__ gba,
                                                         long ldg, int H, int G, int d, int dv,
                                                         const float* __restrict__ neg_a,
                                                         const float* __restrict__ dt_bias, float* __restrict__ state,
                                                         const int* __restrict__ qstart, const int* __restrict__ qlen,
                                                         const int* __restrict__ ctx, const int* __restrict__ rows,
                                                         float* __restrict__ raw) {
  constexpr int DP = 16 * NS;
  __shared__ float qs[DR_TT * DP], ks[DR_TT * DP], vs[DR_TT * DR_COLS], bg[DR_TT * 4];
  const int h = blockIdx.y, s = blockIdx.z;
  const int n = qlen[s];
  if (n <= 0) return;   // the whole workgroup
  const int tid = threadIdx.x, sub = tid & 15, col = tid >> 4;
  const int j0 = blockIdx.x * DR_COLS, j = j0 + col;
  const bool live = j < dv;
  const int kvh = h / (H / G);
  const int q0 = qstart[s], p0 = ctx[s] - n;
  float* sp = state + (((long)rows[s] * H + h) * dv + (live ? j : dv - 1)) * d;
  float S[NS];
#pragma unroll
  for (int r = 0; r < NS; ++r) {
    const int i = sub * NS + r;
    S[r] = (p0 > 0 && live && i < d) ? sp[i] : 0.f;
  }
  const long oq = (long)kvh * d, ok = (long)G * d + (long)kvh * d, ov = 2L * G * d + (long)h * dv;
  const long ob = (long)H * dv + h, oa = (long)H * dv + H + h;
  const float na = neg_a[h], dtb = dt_bias[h], qscale = 1.f / sqrtf((float)d);
  // a group's inputs are fetched into registers one group ahead, so their latency hides under the
  // previous group's recurrence: NS entries of q and of k, one of v, and (lanes < 16) the two logits
  constexpr int NFV = (NS + 7) / 8;          // 16-byte chunks of q (and of k) a thread moves per group: 16 rows of d / 8
  float pq[VL ? 1 : NS], pk[VL ? 1 : NS], pv = 0.f, pb = 0.f, pa = 0.f;
  uint4 vq[VL ? NFV : 1], vk[VL ? NFV : 1];
  const int dch = d >> 3;                    // chunks per row (VL: d % 8 == 0)
  auto fetch = [&](int t0) {
    const int nt = min(DR_TT, n - t0);
    if constexpr (VL) {
#pragma unroll
      for (int f = 0; f < NFV; ++f) {
        const int e = tid + 256 * f;
        const int tt = e / dch, ch = e - tt * dch;
        vq[f] = make_uint4(0u, 0u, 0u, 0u);
        vk[f] = make_uint4(0u, 0u, 0u, 0u);
        if (tt < nt) {
          const u16* row = reinterpret_cast<const u16*>(qkv) + (long)(q0 + t0 + tt) * ldq + 8 * ch;
          vq[f] = *reinterpret_cast<const uint4*>(row + oq);
          vk[f] = *reinterpret_cast<const uint4*>(row + ok);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        const int e = tid + 256 * r;
        const int tt = e / DP, c = e % DP;       // c = r' * 16 + sub'  ->  dim sub' * NS + r'
        const int i = (c & 15) * NS + (c >> 4);
        const bool okx = tt < nt && i < d;
        const T* row = qkv + (long)(q0 + t0 + (okx ? tt : 0)) * ldq;
        pq[r] = okx ? ldf(row + oq + i) : 0.f;
        pk[r] = okx ? ldf(row + ok + i) : 0.f;
      }
    }
    {
      const int tt = tid / DR_COLS, c = tid % DR_COLS;
      pv = (tt < nt && j0 + c < dv) ? ldf(qkv + (long)(q0 + t0 + tt) * ldq + ov + j0 + c) : 0.f;
    }
    if (tid < nt) {
      const T* row = gba + (long)(q0 + t0 + tid) * ldg;
      pb = ldf(row + ob);
      pa = ldf(row + oa);
    }
  };
  if constexpr (VL) {   // dims past d (the lanes' padding) are never written again: zero them once
    for (int e = tid; e < DR_TT * DP; e += 256) { qs[e] = 0.f; ks[e] = 0.f; }
  }
  fetch(0);
  for (int t0 = 0; t0 < n; t0 += DR_TT) {
    const int nt = min(DR_TT, n - t0);
    __syncthreads();   // the previous group is consumed
    if constexpr (VL) {
#pragma unroll
      for (int f = 0; f < NFV; ++f) {
        const int e = tid + 256 * f;
        const int tt = e / dch, ch = e - tt * dch;
        if (tt < DR_TT) {
          float q8[8], k8[8];
          unpack8(vq[f], q8);
          unpack8(vk[f], k8);
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            const int i = 8 * ch + x;          // dim i = sub * NS + r lies at [r * 16 + sub]
            const int pos = tt * DP + (i % NS) * 16 + i / NS;
            qs[pos] = q8[x];
            ks[pos] = k8[x];
          }
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        qs[tid + 256 * r] = pq[r];
        ks[tid + 256 * r] = pk[r];
      }
    }
    vs[tid] = pv;
    if (tid < nt) {
      const float z = pa + dtb;
      const float sp_ = z > 20.f ? z : log1pf(expf(z));
      bg[tid * 4] = 1.f / (1.f + expf(-pb));
      bg[tid * 4 + 1] = expf(na * sp_);
    }
    __syncthreads();
    if (t0 + DR_TT < n) fetch(t0 + DR_TT);
    {   // unit q (times dim^-1/2) and k, and k . q: the 16 lanes of a DPP row take one token
      const int tt = tid >> 4;
      float qv[NS], kv[NS], sq = 0.f, sk = 0.f;
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        qv[r] = qs[tt * DP + r * 16 + sub];
        kv[r] = ks[tt * DP + r * 16 + sub];
        sq += qv[r] * qv[r];
        sk += kv[r] * kv[r];
      }
      sq = row16_sum(sq);
      sk = row16_sum(sk);
      const float rq = qscale / sqrtf(sq + 1e-6f), rk = 1.f / sqrtf(sk + 1e-6f);
      float kq = 0.f;
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        qv[r] *= rq;
        kv[r] *= rk;
        qs[tt * DP + r * 16 + sub] = qv[r];
        ks[tt * DP + r * 16 + sub] = kv[r];
        kq += qv[r] * kv[r];
      }
      kq = row16_sum(kq);
      if (sub == 0) bg[tt * 4 + 2] = kq;
    }
    __syncthreads();
    float o_m = 0.f;
#pragma unroll 4
    for (int u = 0; u < nt; ++u) {   // unrolled: the LDS reads of the next tokens do not depend on the state
      const float beta = bg[u * 4], g = bg[u * 4 + 1], kq = bg[u * 4 + 2], v = vs[u * DR_COLS + col];
      float kk[NS];
      float a2[2] = {0.f, 0.f}, b2[2] = {0.f, 0.f};
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        kk[r] = ks[u * DP + r * 16 + sub];
        a2[r & 1] += S[r] * kk[r];
        b2[r & 1] += S[r] * qs[u * DP + r * 16 + sub];
      }
      const float a = row16_sum(a2[0] + a2[1]);
      const float b = row16_sum(b2[0] + b2[1]);
      const float uu = beta * (v - g * a);
#pragma unroll
      for (int r = 0; r < NS; ++r) S[r] = g * S[r] + kk[r] * uu;
      if (sub == u) o_m = g * b + uu * kq;
    }
    if (live && sub < nt) raw[((long)(q0 + t0 + sub) * H + h) * dv + j] = o_m;
  }
  if (!live) return;
#pragma unroll
  for (int r = 0; r < NS; ++r) {
    const int i = sub * NS + r;
    if (i < d) sp[i] = S[r];
  }
}

__device__ __forceinline__ float pick(bool c, float a, float b) { return c ? a : b; }

// ---- prompt portions: 16 tokens at a time on the matrix cores, in f32.  With S the state before the 16, G_i the sum of the
// decay logarithms up to token i, Gamma_i = exp(G_i) and k, q the unit vectors:
//     A_ij = beta_i exp(G_i - G_j) (k_i . k_j) for j < i,    P_ij = exp(G_i - G_j) (q_i . k_j) for j <= i
//     U = (I + A)^-1 R with R_i = beta_i (v_i - Gamma_i S^T k_i),   O_i = Gamma_i S^T q_i + (P U)_i
//     S <- Gamma S + sum_j exp(G - G_j) k_j u_j^T
// Only R, O and S hang on the state.  delta_prep works out the rest for every 16 tokens at once; delta_tile then walks them.
constexpr int DT_L = 16;          // tokens of a tile
constexpr int DT_P = 20;          // floats from one column of a 16 x 16 tile to the next in LDS: b128 per lane, all banks reached
constexpr int DT_W = 2 * DT_L + 8;  // floats delta_prep leaves per (token, head): a row of (I + A)^-1, a row of P, six scalars

// A wave per (tile, head).  Operands come from the rows as they lie: lane lr of a matrix operand is token lr, and contraction
// step x of lane group g4 stands for dim 16 b + 4 g4 + x, so a lane reads four neighbours.  The inverse is a forward
// substitution with a column per lane (120 multiply-adds; A's columns broadcast from LDS).  8400 tokens of 16 heads of 128: 50 us
// (36 with one chain of d for each dot product, 97 with loads behind branches).
template <typename T, int NB, bool VL>
__global__ void __launch_bounds__(256) delta_prep_kernel(const T* __restrict__ qkv, long ldq, const T* __restrict__ gba, long ldg,
                                                         int H, int G, int d, int dv, const float* __restrict__ neg_a,
                                                         const float* __restrict__ dt_bias, const int* __restrict__ qstart,
                                                         const int* __restrict__ qlen, int S, float* __restrict__ pre) {
  __shared__ __attribute__((aligned(16))) float As4[4][DT_L * DT_P];
  const int tid = threadIdx.x, lr = tid & 15, g4 = (tid >> 4) & 3, w = tid >> 6;
  int s, c;
  if (!dllm::find_chunk<DT_L>(qlen, S, blockIdx.x, s, c)) return;   // the whole workgroup
  const int h = blockIdx.y * 4 + w;
  if (h >= H) return;                                               // the whole wave; no barrier below
  float* As = As4[w];
  const int nt = min(DT_L, qlen[s] - c * DT_L);
  const long tok = (long)qstart[s] + c * DT_L + (lr < nt ? lr : 0);
  f32x4 q[NB], k[NB];
  float sq = 0.f, sk = 0.f;
  {
    const T* x = qkv + tok * ldq + (long)(h / (H / G)) * d;
    const T* y = x + (long)G * d;
    typedef T vec_t __attribute__((ext_vector_type(4)));
    vec_t rq[NB], rk[NB];   // every load in flight before the first is used; places past the row are read elsewhere and dropped
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int i = 16 * b + 4 * g4;
      if constexpr (VL) {
        rq[b] = *reinterpret_cast<const vec_t*>(x + (i < d ? i : 0));
        rk[b] = *reinterpret_cast<const vec_t*>(y + (i < d ? i : 0));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          rq[b][e] = x[i + e < d ? i + e : 0];
          rk[b][e] = y[i + e < d ? i + e : 0];
        }
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = lr < nt && 16 * b + 4 * g4 + e < d;
        const T u = rq[b][e], v = rk[b][e];
        q[b][e] = in ? ldf(&u) : 0.f;
        k[b][e] = in ? ldf(&v) : 0.f;
      }
  }
  float be = 0.f;
  double g = 0.;
  if (lr < nt) {   // decay logarithms summed in 64 bits, so that their differences are exact to 32
    const T* x = gba + tok * ldg + (long)H * dv + h;
    const float z = ldf(x + H) + dt_bias[h];
    const float lg = neg_a[h] * (z > 20.f ? z : log1pf(expf(z)));
    g = lg < -1e5f ? -1e5f : lg;
    be = 1.f / (1.f + expf(-ldf(x)));
  }
#pragma unroll
  for (int o = 1; o < DT_L; o <<= 1) {
    const double x = __shfl_up(g, o, DT_L);
    if (lr >= o) g += x;
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sq += q[b][e] * q[b][e];
      sk += k[b][e] * k[b][e];
    }
  sq = lane_add(sq, 16);
  sk = lane_add(sk, 16);
  sq = lane_add(sq, 32);
  sk = lane_add(sk, 32);
  const float fq = (1.f / sqrtf((float)d)) / sqrtf(sq + 1e-6f), fk = 1.f / sqrtf(sk + 1e-6f);
  // k . k and q . k as sixteen sums of at most eight dims, added pairwise: a chain of d roundings would be the largest error of the rule
  const auto dots = [&](const f32x4(&a)[NB], const f32x4(&b)[NB]) {
    f32x4 p[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) p[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) p[4 * (x & 3) + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x][e], b[x][e], p[4 * (x & 3) + e], 0, 0, 0);
#pragma unroll
    for (int o = 8; o; o >>= 1)
#pragma unroll
      for (int x = 0; x < o; ++x) p[x] += p[x + o];
    return p[0];
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    k[b] *= fk;
    q[b] *= fq;
  }
  const f32x4 kk = dots(k, k), qk = dots(q, k);
  f32x4 av, pv;    // column lr, rows 4 g4 + e
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = 4 * g4 + e;
    const float dec = expf((float)(__shfl(g, i, DT_L) - g));
    const float bi = __shfl(be, i, DT_L);
    av[e] = lr < i ? bi * (dec * kk[e]) : 0.f;
    pv[e] = lr <= i ? dec * qk[e] : 0.f;
  }
  *reinterpret_cast<f32x4*>(As + lr * DT_P + 4 * g4) = av;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float t[DT_L];
#pragma unroll
  for (int i = 0; i < DT_L; ++i) t[i] = i == lr ? 1.f : 0.f;
#pragma unroll
  for (int j = 0; j < DT_L - 1; ++j) {
#pragma unroll
    for (int b = (j + 1) / 4; b < 4; ++b) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(As + j * DT_P + 4 * b);
#pragma unroll
      for (int e = 0; e < 4; ++e) if (4 * b + e > j) t[4 * b + e] -= a[e] * t[j];
    }
  }
  const long base = (long)qstart[s] + c * DT_L;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = 4 * g4 + e;
    float* o = pre + ((base + i) * H + h) * DT_W;
    const float ti = pick(g4 < 2, pick(g4 < 1, t[e], t[4 + e]), pick(g4 < 3, t[8 + e], t[12 + e]));
    if (i < nt) {
      o[lr] = ti;
      o[DT_L + lr] = pv[e];
    }
  }
  const float wd = expf((float)(__shfl(g, DT_L - 1, DT_L) - g)), gam = expf((float)g);
  if (g4 == 0 && lr < nt) {
    float* o = pre + (tok * H + h) * DT_W + 2 * DT_L;
    *reinterpret_cast<f32x4*>(o) = f32x4{gam, be, wd, 0.f};
    *reinterpret_cast<f32x4*>(o + 4) = f32x4{fq, fk, 0.f, 0.f};
  }
}

typedef float f32x3 __attribute__((ext_vector_type(3)));

// A workgroup owns 16 value columns of one (sequence, head); its four waves own a quarter of the key dims each, as the
// accumulators of the last product, which are at once the right operand of S^T k and S^T q.  The waves' parts meet in LDS, a
// thread sums one element of each, and U = (I + A)^-1 R comes out as the right operand of the state's update.  Serial over the
// tiles, so the chain of one tile bounds it: two products, one exchange, two small products, the update.  Sums of more than four terms go in
// parts that are added pairwise, or the largest last.  Three workgroups of the wide-load form fit a CU (its registers are bounded for
// that: with two, 6 sequences are a second pass and take 437 us).  bf16, 16 heads of 128 x 128, with the two launches beside it: 6
// sequences of 1400 tokens 373 us, one of 4096 tokens 433 (421 and 535 with waits for loads just issued, 617 and 1219 token by token).
// f32 errors against 64 bits over 385 tokens, state and outputs, token by token
// in brackets: decays near 1 1.5e-7 (5.6e-7), 1.7e-7 (2.6e-7); a model's (0.01 to 0.3 a token) 1.2e-7 (1.9e-7), 1.6e-7 (1.7e-7); up
// to 4 a token 1.0e-7 (1.05e-7), 1.53e-7 (1.49e-7).
template <typename T, int NS, bool VL>
__global__ void __launch_bounds__(256, VL ? 3 : 2) delta_tile_kernel(const T* __restrict__ qkv, long ldq, int H, int G, int d, int dv,
                                                         float* __restrict__ state, const int* __restrict__ qstart,
                                                         const int* __restrict__ qlen, const int* __restrict__ ctx,
                                                         const int* __restrict__ rows, const float* __restrict__ pre,
                                                         float* __restrict__ raw) {
  constexpr int KD = 16 * NS, LD = KD + 4, NB = KD / 64;   // NB blocks of 16 dims a wave
  constexpr int TP = DT_L * DT_P;
  typedef T row_t __attribute__((ext_vector_type(NS)));
  __shared__ __attribute__((aligned(16))) float qs[2][DT_L * LD], ks[2][DT_L * LD], part[4 * 2 * TP];
  __shared__ __attribute__((aligned(16))) float Rs[TP], Os[TP], ws[DT_L];
  __shared__ float last;
  const int h = blockIdx.y, s = blockIdx.z;
  const int n = qlen[s];
  if (n <= 0) return;   // the whole workgroup
  const int tid = threadIdx.x, lr = tid & 15, row = tid >> 4, w = __builtin_amdgcn_readfirstlane(tid >> 6), g4 = (tid >> 4) & 3;
  const int j = blockIdx.x * 16 + lr;
  const bool live = j < dv;
  const int q0 = qstart[s], p0 = ctx[s] - n;
  const bool vs = (d & 3) == 0 && ((uintptr_t)state & 15) == 0;
  float* sp = state + (((long)rows[s] * H + h) * dv + (live ? j : dv - 1)) * d;
  f32x4 S[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int i = 16 * (w * NB + b) + 4 * g4;
    S[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p0 > 0 && live) {
      if (vs) {
        if (i < d) S[b] = *reinterpret_cast<const f32x4*>(sp + i);
      } else {
#pragma unroll
        for (int x = 0; x < 4; ++x) if (i + x < d) S[b][x] = sp[i + x];
      }
    }
  }
  const long oq = (long)(h / (H / G)) * d, ok = (long)G * d + oq, ov = 2L * G * d + (long)h * dv + (live ? j : dv - 1);
  // two tiles' inputs travel while one is computed: NS dims of one token's q and k with their factors; one value and its
  // scalars, four entries of a row of (I + A)^-1 and of P.  No load stands behind a condition or is copied on from tile to tile (rows past
  // the end read the last token's and become zeros where they are used; two tiles take turns with two sets of registers): the
  // compiler then knows which are in flight, where it waited for all of them at the head of every tile
  const int kcol = NS * lr < d ? NS * lr : 0;
  row_t rq, rk;
  float2 fac = make_float2(0.f, 0.f);
  auto fetch_keys = [&](int t0) {
    const int at = q0 + min(t0 + row, n - 1);
    const T* x = qkv + (long)at * ldq;
    if constexpr (VL) {
      rq = *reinterpret_cast<const row_t*>(x + oq + kcol);
      rk = *reinterpret_cast<const row_t*>(x + ok + kcol);
    } else {
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        rq[r] = x[oq + min(kcol + r, d - 1)];
        rk[r] = x[ok + min(kcol + r, d - 1)];
      }
    }
    fac = *reinterpret_cast<const float2*>(pre + ((long)at * H + h) * DT_W + 2 * DT_L + 4);
  };
  auto stage_keys = [&](int buf, int t0) {
    const bool in = t0 + row < n;
#pragma unroll
    for (int r = 0; r < NS; r += 4) {
      f32x4 a, b;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const T y = rq[r + x], z = rk[r + x];
        const bool on = in && NS * lr + r + x < d;
        a[x] = on ? ldf(&y) * fac.x : 0.f;
        b[x] = on ? ldf(&z) * fac.y : 0.f;
      }
      *reinterpret_cast<f32x4*>(qs[buf] + row * LD + NS * lr + r) = a;
      *reinterpret_cast<f32x4*>(ks[buf] + row * LD + NS * lr + r) = b;
    }
  };
  // (three scalars: a register that a load writes and nobody reads is given away while the load is under way, and its next owner waits)
  struct Tile { T v; f32x3 sc; f32x4 inv, p; };
  auto fetch_tile = [&](Tile& t, int t0) {
    const int at = q0 + min(t0 + row, n - 1);
    t.v = qkv[(long)at * ldq + ov];
    t.sc = *reinterpret_cast<const f32x3*>(pre + ((long)at * H + h) * DT_W + 2 * DT_L);
    const float* x = pre + ((long)(q0 + min(t0 + lr, n - 1)) * H + h) * DT_W + 4 * g4;
    t.inv = *reinterpret_cast<const f32x4*>(x);
    t.p = *reinterpret_cast<const f32x4*>(x + DT_L);
  };
  __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): the state has landed, so that no tile waits for it
  fetch_keys(0);
  Tile even, odd;
  fetch_tile(even, 0);
  fetch_tile(odd, DT_L);
  stage_keys(0, 0);
  fetch_keys(DT_L);
  __syncthreads();
  auto tile = [&](const int t0, const int buf, Tile& cur) {
    const int nt = min(DT_L, n - t0);
    {
      f32x4 tk[4], tq[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) tk[x] = tq[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int i = lr * LD + 16 * (w * NB + b) + 4 * g4;
        const f32x4 a = *reinterpret_cast<const f32x4*>(ks[buf] + i), q = *reinterpret_cast<const f32x4*>(qs[buf] + i);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          tk[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], S[b][x], tk[x], 0, 0, 0);
          tq[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[x], S[b][x], tq[x], 0, 0, 0);
        }
      }
      float* p = part + w * 2 * TP + lr * DT_P + 4 * g4;
      *reinterpret_cast<f32x4*>(p) = (tk[0] + tk[1]) + (tk[2] + tk[3]);
      *reinterpret_cast<f32x4*>(p + TP) = (tq[0] + tq[1]) + (tq[2] + tq[3]);
    }
    __syncthreads();
    if (nt < DT_L) {      // the last tile: zeros behind the end
      if (row >= nt) cur.sc = f32x3{0.f, 0.f, 0.f};
      if (lr >= nt) cur.inv = cur.p = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    {   // token `row`, column lr
      const float* p = part + lr * DT_P + row;
      const float ek = (p[0] + p[2 * TP]) + (p[4 * TP] + p[6 * TP]), eq = (p[TP] + p[3 * TP]) + (p[5 * TP] + p[7 * TP]);
      Rs[lr * DT_P + row] = row < nt ? cur.sc[1] * (ldf(&cur.v) - cur.sc[0] * ek) : 0.f;
      Os[lr * DT_P + row] = cur.sc[0] * eq;
      if (lr == 0) ws[row] = cur.sc[2];
      if (tid == 16 * (nt - 1)) last = cur.sc[0];
    }
    stage_keys(buf ^ 1, t0 + DT_L);      // (behind the last tile: zeros that nobody reads)
    fetch_keys(t0 + 2 * DT_L);
    __syncthreads();
    f32x4 r = *reinterpret_cast<const f32x4*>(Rs + lr * DT_P + 4 * g4);
    // An infinity or NaN of a token must not reach those before it, whose zeros in (I + A)^-1 and P it would meet: it leaves the
    // products, and the column is NaN from its first such row on.
    int lost = DT_L;
    const bool bad = __ballot(!(fmaf(r[1], 0.f, r[0] * 0.f) + fmaf(r[3], 0.f, r[2] * 0.f) == 0.f));
    if (bad) {
#pragma unroll
      for (int e = 3; e >= 0; --e)
        if (!(r[e] * 0.f == 0.f)) {
          lost = 4 * g4 + e;
          r[e] = 0.f;
        }
      lost = min(lost, lane_xor(lost, 16));
      lost = min(lost, lane_xor(lost, 32));
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 u4[4];
    // each of the small products as four sums: token i's own term, which steep decays leave alone, is then the last of sum i % 4 (of
    // entry e = i % 4 of this lane's rows 4 g4 + e), and that sum is added last
    const f32x4 we = *reinterpret_cast<const f32x4*>(ws + 4 * g4);
    const float gam = last;
#pragma unroll
    for (int x = 0; x < 4; ++x) u4[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.inv[x], r[x], zero, 0, 0, 0);
    f32x4 u;
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = (u4[e ^ 1][e] + (u4[e ^ 2][e] + u4[e ^ 3][e])) + u4[e][e];
    f32x4 z = we * u;
    if (bad) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z[e] = 4 * g4 + e < lost ? z[e] : __builtin_nanf("");
        u[e] = 4 * g4 + e < lost ? u[e] : 0.f;
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float* kp = ks[buf] + 4 * g4 * LD + 16 * (w * NB + b) + lr;
      f32x4 s4[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) s4[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(kp[x * LD], z[x], zero, 0, 0, 0);
      S[b] = ((gam * S[b] + (s4[0] + s4[1])) + s4[2]) + s4[3];      // the last tokens last
    }
    if (w == ((t0 >> 4) & 3)) {   // the waves take turns with the outputs
      f32x4 o4[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) o4[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.p[x], u[x], zero, 0, 0, 0);
      f32x4 o = *reinterpret_cast<const f32x4*>(Os + lr * DT_P + 4 * g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (o[e] + (o4[e ^ 1][e] + (o4[e ^ 2][e] + o4[e ^ 3][e]))) + o4[e][e];
      if (bad)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = 4 * g4 + e < lost ? o[e] : __builtin_nanf("");
#pragma unroll
      for (int x = 0; x < 4; ++x)
        if (live && 4 * g4 + x < nt) raw[((long)(q0 + t0 + 4 * g4 + x) * H + h) * dv + j] = o[x];
    }
    fetch_tile(cur, t0 + 2 * DT_L);
  };
  // pairs of tiles and perhaps one more: a way out between two of a pair would meet the way back in a block, with its loads under way
  const int tiles = (n + DT_L - 1) / DT_L;
  for (int i = 0; i < tiles / 2; ++i) {
    tile(2 * i * DT_L, 0, even);
    tile((2 * i + 1) * DT_L, 1, odd);
  }
  if (tiles & 1) tile((tiles - 1) * DT_L, 0, even);
  if (!live) return;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int i = 16 * (w * NB + b) + 4 * g4;
    if (vs) {
      if (i < d) *reinterpret_cast<f32x4*>(sp + i) = S[b];
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) if (i + x < d) sp[i + x] = S[b][x];
    }
  }
}

// is `tok` a token of one of the S sequences?  (the tokens a captured step is padded with are of none)  Every lane of the wave asks.
__device__ __forceinline__ bool any_seq(const int* qstart, const int* qlen, int S, long tok, int lane, int width) {
  bool in = false;
  for (int s = lane; s < S; s += width) {
    const int a = qstart[s];
    in |= tok >= a && tok < a + qlen[s];
  }
  for (int o = width >> 1; o; o >>= 1) in |= __shfl_xor((int)in, o) != 0;
  return in;
}

// out = raw / rms(raw over dv) * w * silu(gate).  A row is one (token, head): LPR lanes on it with four values a lane at a time
// (V4: rows of whole, aligned vectors), or a wave with one.  Memory bounds it: 8400 tokens of 16 heads of 128 in 41 us
// (67 us with a value a lane and every lane looking through the sequences).
template <typename T, int LPR, bool V4>
__global__ void __launch_bounds__(256) delta_finish_kernel(const float* __restrict__ raw, const T* __restrict__ gba, long ldg,
                                                           int H, int dv, const float* __restrict__ w, float eps,
                                                           const int* __restrict__ qstart, const int* __restrict__ qlen,
                                                           int S, T* __restrict__ out, long rows_total) {
  constexpr int W = V4 ? 4 : 1;
  typedef T vec_t __attribute__((ext_vector_type(W)));
  typedef float vecf_t __attribute__((ext_vector_type(W)));
  const long rr = (long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const int lane = threadIdx.x % LPR;
  const long r = rr < rows_total ? rr : rows_total - 1;
  const long tok = r / H;
  const int h = (int)(r % H);
  const bool live = any_seq(qstart, qlen, S, tok, lane, LPR);   // tokens of no sequence become zeros
  const float* o = raw + r * dv;
  const T* gp = gba + tok * ldg + (long)h * dv;
  T* y = out + tok * ((long)H * dv) + (long)h * dv;
  float ss = 0.f;
  for (int j = lane * W; j < dv; j += LPR * W) {
    const vecf_t v = *reinterpret_cast<const vecf_t*>(o + j);
#pragma unroll
    for (int x = 0; x < W; ++x) ss += v[x] * v[x];
  }
#pragma unroll
  for (int x = LPR >> 1; x; x >>= 1) ss = lane_add(ss, x);
  const float rs = 1.f / sqrtf(ss / (float)dv + eps);
  if (rr >= rows_total) return;
  for (int j = lane * W; j < dv; j += LPR * W) {
    const vecf_t v = *reinterpret_cast<const vecf_t*>(o + j);
    const vec_t g = *reinterpret_cast<const vec_t*>(gp + j);
    vec_t res;
#pragma unroll
    for (int x = 0; x < W; ++x) {
      const T gx = g[x];
      const float z = ldf(&gx);
      T q;
      stf(&q, live ? v[x] * rs * w[j + x] * (z / (1.f + expf(-z))) : 0.f);
      res[x] = q;
    }
    *reinterpret_cast<vec_t*>(y + j) = res;
  }
}

template <typename T>
int launch_finish(const float* raw, const T* gba, long ldg, int H, int dv, const float* w, float eps, const int* qstart,
                  const int* qlen, int S, T* out, long rows, hipStream_t st) {
  const bool v4 = dv % 4 == 0 && ldg % 4 == 0 && (((uintptr_t)gba | (uintptr_t)out) & (4 * sizeof(T) - 1)) == 0;
#define FIN(LPR, V4) \
  hipLaunchKernelGGL((delta_finish_kernel<T, LPR, V4>), dim3((unsigned)((rows + 256 / LPR - 1) / (256 / LPR))), dim3(256), 0, st, raw, gba, \
                     ldg, H, dv, w, eps, qstart, qlen, S, out, rows)
  if (!v4) FIN(64, false); else if (dv <= 64) FIN(16, true); else if (dv <= 128) FIN(32, true); else FIN(64, true);
#undef FIN
  return (int)hipGetLastError();
}

template <typename T, bool VL>
int launch_delta(int ns, float* pre, long total, dim3 g, hipStream_t st, const T* qkv, long ldq, const T* gba, long ldg, int H, int G, int d, int dv,
                 const float* neg_a, const float* dt_bias, float* state, const int* qstart, const int* qlen, const int* ctx,
                 const int* rows, float* raw) {
#define DELTA(NS) hipLaunchKernelGGL((delta_rule_kernel<T, NS, (VL && sizeof(T) == 2)>), g, dim3(256), 0, st, qkv, ldq, gba, ldg, H, G, d, dv, neg_a, dt_bias, state, qstart, qlen, ctx, rows, raw)
  if (pre) {
#define TILE(NS) \
  hipLaunchKernelGGL((delta_prep_kernel<T, NS, VL>), dim3((unsigned)(total / DT_L + g.z), (H + 3) / 4), dim3(256), 0, st, qkv, ldq, gba, ldg, \
                     H, G, d, dv, neg_a, dt_bias, qstart, qlen, (int)g.z, pre); \
  hipLaunchKernelGGL((delta_tile_kernel<T, NS, VL>), g, dim3(256), 0, st, qkv, ldq, H, G, d, dv, state, qstart, qlen, ctx, rows, pre, raw)
    if (ns <= 4) { TILE(4); } else { TILE(8); }
#undef TILE
    return (int)hipGetLastError();
  }
  if (ns <= 1) DELTA(1); else if (ns <= 2) DELTA(2); else if (ns <= 4) DELTA(4); else if (ns <= 8) DELTA(8); else DELTA(16);
#undef DELTA
  return (int)hipGetLastError();
}

}  // namespace

// floats of scratch per (token, head) with which dllm_delta_rule takes 16 tokens at a time; 0: it goes token by token
extern "C" int dllm_delta_pre(int d) { return d <= 128 ? DT_W : 0; }

// qkv [T, 2 G d + H dv] (q | k | v after convolution and SiLU), gba [T, H dv + 2 H] (gate | beta |
// decay logits), state [slots, H, dv, d] f32, raw [T, H, dv] f32 scratch, out [T, H dv].
extern "C" int dllm_delta_rule(const void* qkv, long ldq, const void* gba, long ldg, int f32, int H, int G, int d, int dv,
                               const float* neg_a, const float* dt_bias, const float* norm_w, float eps, float* state,
                               const int* qstart, const int* qlen, const int* ctx, const int* rows, float* raw, void* out,
                               int S, long T, float* pre, hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (d < 1 || d > 256 || G < 1 || H % G || (pre && d > 128)) return -1;
  const int ns = (d + 15) / 16;
  const dim3 g((dv + DR_COLS - 1) / DR_COLS, H, S);
  const long rows_total = T * H;
  int rc;
  // 16-byte row vectors: every q / k head starts on a 16-byte boundary of a 16-byte aligned row
  const bool vl = d % 8 == 0 && ldq % 8 == 0 && ((uintptr_t)qkv & 15) == 0;
  if (f32) {
    rc = vl && pre ? launch_delta<float, true>(ns, pre, T, g, st, (const float*)qkv, ldq, (const float*)gba, ldg, H, G, d, dv, neg_a,
                                                 dt_bias, state, qstart, qlen, ctx, rows, raw)
                     : launch_delta<float, false>(ns, pre, T, g, st, (const float*)qkv, ldq, (const float*)gba, ldg, H, G, d, dv, neg_a,
                                                  dt_bias, state, qstart, qlen, ctx, rows, raw);
    if (!rc) rc = launch_finish<float>(raw, (const float*)gba, ldg, H, dv, norm_w, eps, qstart, qlen, S, (float*)out, rows_total, st);
  } else {
    if (vl)
      rc = launch_delta<u16, true>(ns, pre, T, g, st, (const u16*)qkv, ldq, (const u16*)gba, ldg, H, G, d, dv, neg_a, dt_bias, state,
                                   qstart, qlen, ctx, rows, raw);
    else
      rc = launch_delta<u16, false>(ns, pre, T, g, st, (const u16*)qkv, ldq, (const u16*)gba, ldg, H, G, d, dv, neg_a, dt_bias, state,
                                    qstart, qlen, ctx, rows, raw);
    if (!rc) rc = launch_finish<u16>(raw, (const u16*)gba, ldg, H, dv, norm_w, eps, qstart, qlen, S, (u16*)out, rows_total, st);
  }
  return rc;
}
