// Memory-bound elementwise / small-reduction kernels (all 16-B vectorised, f32 math):
//   silu_mul     : out[t, i] = silu(gu[t, i]) * gu[t, I + i]        (SwiGLU, fused gate|up GEMM output)
//   gelu         : y = 0.5 x (1 + erf(x / sqrt 2))                    (MiniLM FFN)
//   mean_pool_l2 : out[b] = normalize(sum_s mask[b,s] x[b,s,:] / sum_s mask[b,s])   (sentence embedding)
//   moe_gate_topk: softmax over E experts, top-k, renormalised weights (Mixtral routing)
//   embed        : out[t] = table[ids[t] - lo] if lo <= ids[t] < lo + rows else 0   (token embedding;
//                  the masked form is the vocab-parallel shard of a TP rank, summed by the all-reduce)
#include "common.h"

namespace {

__global__ void silu_mul_kernel(const u16* __restrict__ gu, u16* __restrict__ out, long T, int I, long in_stride) {
  // 32-bit index math (the launcher guarantees T * I / 8 < 2^30, so v + stride cannot overflow): a 64-bit divide is a long
  // software sequence on CDNA, a 32-bit one a handful of VALU ops
  const int nv = I >> 3;
  const int nvec = (int)(T * nv);
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < nvec; v += gridDim.x * blockDim.x) {
    const int t = v / nv;
    const int c = (v - t * nv) * 8;
    float gf[8], uf[8], o[8];
    unpack8(ld16(gu + t * in_stride + c), gf);
    unpack8(ld16(gu + t * in_stride + I + c), uf);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = gf[j] / (1.f + __expf(-gf[j])) * uf[j];
    st16(out + t * (long)I + c, pack8(o));
  }
}

// one wave per token row, 16-B vectors; rows of a 288 GB-resident table are gathered straight to
// registers (a random-row gather reads at ~5.5 TB/s: MI355X_MICROARCH.md)
// ssq (optional): the row's sum of squares, ssq[t] — the first decoder layer's folded-RMSNorm row
// scale then needs no separate res_add_ssq pass over the embeddings (one launch less per step)
// sc_buf != nullptr: the LAST workgroup instead applies a decode step's block-table updates
// (scatter_pairs_kernel's job: dst[idx_i] = val_i for sc_buf = [n, idx0, val0, ...]), so a decode
// step starts with one launch instead of two (~4.5 us at batch 1, profiles/r3_single_stream_decode.md)
__global__ void __launch_bounds__(256) embed_kernel(const int* __restrict__ ids, const u16* __restrict__ table,
                                                    u16* __restrict__ out, long T, int H, long lo, long rows,
                                                    float* __restrict__ ssq, int* __restrict__ sc_dst,
                                                    const int* __restrict__ sc_buf, int sc_cap) {
  if (sc_buf != nullptr && blockIdx.x == gridDim.x - 1) {
    const int n = min(sc_buf[0], sc_cap);
    for (int i = threadIdx.x; i < n; i += blockDim.x) sc_dst[sc_buf[1 + 2 * i]] = sc_buf[2 + 2 * i];
    return;
  }
  const long t = blockIdx.x * 4L + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= T) return;
  const long r = ids[t] - lo;
  const bool ok = r >= 0 && r < rows;
  const u16* src = table + (ok ? r : 0) * (long)H;
  u16* dst = out + t * (long)H;
  float s = 0.f;
  for (int c = (threadIdx.x & 63) * 8; c < H; c += 64 * 8) {
    const uint4 v = ok ? ld16(src + c) : make_uint4(0, 0, 0, 0);
    st16(dst + c, v);
    if (ssq) {
      float f[8];
      unpack8(v, f);
#pragma unroll
      for (int j = 0; j < 8; ++j) s += f[j] * f[j];
    }
  }
  if (ssq) {
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) ssq[t] = s;
  }
}

__global__ void gelu_kernel(const u16* __restrict__ x, u16* __restrict__ y, long n8) {
  for (long v = blockIdx.x * (long)blockDim.x + threadIdx.x; v < n8; v += (long)gridDim.x * blockDim.x) {
    float f[8];
    unpack8(ld16(x + v * 8), f);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = gelu_bf(f[j]);
    st16(y + v * 8, pack8(f));
  }
}

// A workgroup per text; rows as 16-byte vectors, the workgroup's 256 / (H / 8) row groups side by side and four rows a group in
// flight, met in LDS.  96 texts of up to 72 tokens x 384: 7 us (56 with two-byte loads and one row at a time).  starts: text b's
// rows begin at row starts[b] of a packed batch of T rows, else at b S.
__global__ void __launch_bounds__(256) mean_pool_l2_kernel(const u16* __restrict__ x, const int* __restrict__ lens,
                                                           float* __restrict__ out, int S, int H,
                                                           const int* __restrict__ starts, int T) {
  __shared__ float red[16];
  extern __shared__ float part[];      // [row groups][H]
  const int b = blockIdx.x, nv = H >> 3, G = 256 / nv, v = threadIdx.x % nv, g = threadIdx.x / nv;
  const long row0 = starts ? min(max(starts[b], 0), T) : (long)b * S;
  const int n = starts ? (int)min((long)max(lens[b], 0), T - row0) : lens[b];
  const u16* xr = x + row0 * H + 8 * v;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (g < G) {
    for (int s = g; s < n; s += 4 * G) {
      uint4 r[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) r[u] = ld16(xr + (long)min(s + u * G, n - 1) * H);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float f[8];
        unpack8(r[u], f);
        if (s + u * G < n)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] += f[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) part[g * H + 8 * v + e] = acc[e];
  }
  __syncthreads();
  float y[8], ss = 0.f;                // H <= 2048: at most 8 columns a thread
  const float inv = n > 0 ? 1.f / n : 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int h = threadIdx.x + 256 * i;
    y[i] = 0.f;
    if (h < H) {
      for (int gg = 0; gg < G; ++gg) y[i] += part[gg * H + h];
      y[i] *= inv;
    }
    ss += y[i] * y[i];
  }
  const float nrm = sqrtf(block_sum(ss, red));
  const float sc = 1.f / fmaxf(nrm, 1e-12f);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int h = threadIdx.x + 256 * i;
    if (h < H) out[(long)b * H + h] = y[i] * sc;
  }
}

// The same behind a LayerNorm (norm.hip's arithmetic, each row rounded as it leaves there), rows of at most 512: eight waves a text, each with four
// rows in flight.  96 texts of up to 72 tokens x 384: 7.1 us, the two launches 11.2; one text of 12: 3.3.
__global__ void __launch_bounds__(512) ln_pool_l2_kernel(const u16* __restrict__ x, const u16* __restrict__ w, const u16* __restrict__ bias, float eps,
                                                         const int* __restrict__ lens, float* __restrict__ out, int H, const int* __restrict__ starts,
                                                         int T) {
  constexpr int NW = 8;
  __shared__ float red[16];
  __shared__ __attribute__((aligned(16))) float part[NW][512];
  const int b = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = 8 * lane;
  const int row0 = min(max(starts[b], 0), T), n = min(max(lens[b], 0), T - row0);
  const bool on = c < H;
  const u16* xr = x + (long)row0 * H + (on ? c : 0);
  float gw[8], gb[8], acc[8] = {};
  unpack8(on ? ld16(w + c) : make_uint4(0u, 0u, 0u, 0u), gw);
  unpack8(on ? ld16(bias + c) : make_uint4(0u, 0u, 0u, 0u), gb);
  for (int s = wave; s < n; s += 4 * NW) {
    uint4 r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = ld16(xr + (long)min(s + u * NW, n - 1) * H);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s + u * NW >= n) break;      // (uniform)
      float v[8], sum = 0.f, q = 0.f, o[8];
      unpack8(on ? r[u] : make_uint4(0u, 0u, 0u, 0u), v);
#pragma unroll
      for (int j = 0; j < 8; ++j) sum += v[j];
      const float mean = wave_sum(sum) / H;
      if (on)
#pragma unroll
        for (int j = 0; j < 8; ++j) { const float d = v[j] - mean; q += d * d; }
      const float rstd = rsqrtf(wave_sum(q) / H + eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[j] - mean) * rstd * gw[j] + gb[j];
      unpack8(pack8(o), o);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += o[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) part[wave][c + j] = acc[j];
  __syncthreads();
  float y = 0.f;
  if ((int)threadIdx.x < H) {
#pragma unroll
    for (int g = 0; g < NW; ++g) y += part[g][threadIdx.x];
    y *= n > 0 ? 1.f / n : 0.f;
  }
  const float sc = 1.f / fmaxf(sqrtf(block_sum(y * y, red)), 1e-12f);
  if ((int)threadIdx.x < H) out[(long)b * H + threadIdx.x] = y * sc;
}

// widths that are no whole vectors (H <= 1024)
__global__ void __launch_bounds__(256) mean_pool_any_kernel(const u16* __restrict__ x, const int* __restrict__ lens,
                                                            float* __restrict__ out, int S, int H,
                                                            const int* __restrict__ starts, int T) {
  __shared__ float red[16];
  const int b = blockIdx.x;
  const long row0 = starts ? min(max(starts[b], 0), T) : (long)b * S;
  const int n = starts ? (int)min((long)max(lens[b], 0), T - row0) : lens[b];
  float acc[4] = {0.f, 0.f, 0.f, 0.f};  // H <= 4 * blockDim
  for (int s = 0; s < n; ++s) {
    const u16* row = x + (row0 + s) * H;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int h = threadIdx.x + i * blockDim.x;
      if (h < H) acc[i] += bf2f(row[h]);
    }
  }
  float ss = 0.f;
  const float inv = n > 0 ? 1.f / n : 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) { acc[i] *= inv; ss += acc[i] * acc[i]; }
  const float nrm = sqrtf(block_sum(ss, red));
  const float sc = 1.f / fmaxf(nrm, 1e-12f);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int h = threadIdx.x + i * blockDim.x;
    if (h < H) out[(long)b * H + h] = acc[i] * sc;
  }
}

// one thread per token; E <= 64, k <= 8
__global__ void moe_gate_kernel(const float* __restrict__ logits, int T, int E, int k, int* __restrict__ ids,
                                float* __restrict__ w) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  const float* l = logits + (long)t * E;
  unsigned long long used = 0ull;
  float sel[8];
  int sid[8];
  for (int i = 0; i < k; ++i) {
    float best = -INFINITY;
    int bi = 0;
    for (int e = 0; e < E; ++e)
      if (!((used >> e) & 1ull) && l[e] > best) { best = l[e]; bi = e; }
    used |= 1ull << bi;
    sel[i] = best;
    sid[i] = bi;
  }
  // softmax over all E then renormalise over the selected == softmax over the selected logits
  const float m = sel[0];
  float s = 0.f;
  for (int i = 0; i < k; ++i) { sel[i] = __expf(sel[i] - m); s += sel[i]; }
  for (int i = 0; i < k; ++i) { ids[(long)t * k + i] = sid[i]; w[(long)t * k + i] = sel[i] / s; }
}
// A token's choice from its logits (lane e: expert e's; one wave): the k largest, the lower expert first among equals; NaN is never chosen, and
// expert 0 where nothing is left to choose.  Softmax over all E then renormalise over the selected == softmax over the selected logits;
// summed in the order of choice.  `o`: the token's first pair
__device__ __forceinline__ void router_choice(float lg, int lane, int E, int k, long o, int* ids, float* w, int shared, float scale) {
  float left = lane < E && lg > -INFINITY ? lg : -INFINITY, sel = -INFINITY;
  int sid = 0;
  for (int i = 0; i < k; ++i) {
    float best = left;
    int bi = lane;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const float ov = lane_xor(best, m);
      const int oi = lane_xor(bi, m);
      if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
    }
    if (!(best > -INFINITY)) bi = 0;
    if (lane == i) { sel = best; sid = bi; }
    if (lane == bi) left = -INFINITY;
  }
  const float ex = __expf(sel - __shfl(sel, 0));
  float sum = 0.f;
  for (int i = 0; i < k; ++i) sum += __shfl(ex, i);
  if (lane < k) { ids[o + lane] = sid; w[o + lane] = ex / sum * scale; }
  if (shared && lane == k) { ids[o + k] = E; w[o + k] = 1.f; }
}

// Fused router: logits[t, e] = x[t] . wg[e] in fp32 (one wave per token: each lane holds XC 8-wide
// chunks of its token's row in registers, every expert's dot product is summed in a fixed order and
// reduced with an xor butterfly), then the same top-k / renormalised softmax as moe_gate_kernel.
// A token's result depends only on its own row, never on how many tokens share the launch, so a
// padded graph batch routes exactly like an eager one (a vendor GEMM picks its reduction split by M).
// The weights are multiplied by ``scale``; with ``shared`` every token gets one more pair, expert E with
// weight 1 (a shared expert stored behind the routed ones).
// Bound by latency: the rows' loads, one butterfly per expert (they overlap) and the choice.  Lane e holds expert e's logit and the
// choice is a wave-wide maximum (a lane walking the logits in LDS with its choices in scratch took most of the launch): 8
// experts, width 1024, 24 tokens 6.0 us against 10.0 (an empty launch shows 3).
// NORM: x is the residual stream; the wave first norms its row, bf16(x / rms(x) * norm_w), leaves that in xn and routes it.
template <int XC, int EB, bool NORM>   // EB experts' rows in flight
__global__ void __launch_bounds__(256) moe_router_kernel(const u16* __restrict__ x, long x_stride,
                                                         const u16* __restrict__ wg, int T, int E, int H, int k,
                                                         int* __restrict__ ids, float* __restrict__ w,
                                                         float* __restrict__ logits, int shared, float scale,
                                                         const u16* __restrict__ norm_w, float eps, u16* __restrict__ xn) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.x * 4 + wv;
  if (t >= T) return;  // whole wave; no block barrier below
  const int nc = H >> 3;
  // no load stands behind a condition (chunks past the row read its last and become zeros, experts past the last read its row and are
  // not chosen): us in a captured graph, 24 rows of 1024 and 8 experts 3.9 -> 3.7, of 2048 5.0 -> 4.7, 64 experts 21.2 -> 16.7
  // (with the norm 4.3, 5.6 -> 5.5, 21.9 -> 17.4), 3000 rows of 1024 5.8 -> 5.5 (7.5 -> 6.9).  The first
  // experts' rows beside the token's instead of behind it gained nothing
  uint4 xr[XC], nw[NORM ? XC : 1];
#pragma unroll
  for (int c = 0; c < XC; ++c) {
    const int ch = min(lane + 64 * c, nc - 1);
    xr[c] = ld16(x + (long)t * x_stride + 8 * ch);
    if constexpr (NORM) nw[c] = ld16(norm_w + 8 * ch);
  }
#pragma unroll
  for (int c = 0; c < XC; ++c)
    if (lane + 64 * c >= nc) {
      xr[c] = make_uint4(0u, 0u, 0u, 0u);
      if constexpr (NORM) nw[c] = xr[c];
    }
  if constexpr (NORM) {
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < XC; ++c) {
      float f[8];
      unpack8(xr[c], f);
#pragma unroll
      for (int q = 0; q < 8; ++q) s += f[q] * f[q];
    }
    const float rstd = rsqrtf(wave_sum(s) / H + eps);
#pragma unroll
    for (int c = 0; c < XC; ++c) {
      const int ch = lane + 64 * c;
      float f[8], g[8];
      unpack8(xr[c], f);
      unpack8(nw[c], g);
#pragma unroll
      for (int q = 0; q < 8; ++q) f[q] = f[q] * rstd * g[q];
      xr[c] = pack8(f);
      if (ch < nc) st16(xn + (long)t * H + 8 * ch, xr[c]);
    }
  }
  float lg = -INFINITY;   // lane e: expert e's logit
  for (int e0 = 0; e0 < E; e0 += EB) {
    uint4 wr[EB][XC];
#pragma unroll
    for (int y = 0; y < EB; ++y)
#pragma unroll
      for (int c = 0; c < XC; ++c) wr[y][c] = ld16(wg + (long)min(e0 + y, E - 1) * H + 8 * min(lane + 64 * c, nc - 1));
    if (nc < 64 * XC) {      // (uniform)
#pragma unroll
      for (int c = 0; c < XC; ++c)
        if (lane + 64 * c >= nc)
#pragma unroll
          for (int y = 0; y < EB; ++y) wr[y][c] = make_uint4(0u, 0u, 0u, 0u);
    }
    float s[EB];
#pragma unroll
    for (int x = 0; x < EB; ++x) {
      s[x] = 0.f;
#pragma unroll
      for (int c = 0; c < XC; ++c) {
        float f[8], g[8];
        unpack8(wr[x][c], f);
        unpack8(xr[c], g);
#pragma unroll
        for (int q = 0; q < 8; ++q) s[x] += g[q] * f[q];
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1)
#pragma unroll
      for (int x = 0; x < EB; ++x) s[x] = lane_add(s[x], m);
#pragma unroll
    for (int x = 0; x < EB; ++x) lg = lane == e0 + x ? s[x] : lg;
  }
  if (logits != nullptr && lane < E) logits[(long)t * E + lane] = lg;
  router_choice(lg, lane, E, k, (long)t * (k + shared), ids, w, shared, scale);
}

// norm_resadd (seqmix.hip, one group: x += rmsnorm(y + bias) * w, xl = the rounded stream) and the router of that row: a workgroup a token, the
// row's entries and sums as norm_resadd_reg_kernel has them, then two experts a wave at a time with moe_router_kernel's sums, the
// first two's rows asked for beside the token's.  Both launches were latency: us in a captured graph, two / here, width 1024, 8 experts:
// 1 token 5.6 / 3.6, 24 6.4 / 3.9, 300 6.9 / 4.5, 4000 15.6 / 12.4; 64 experts 24 tokens 13.4 / 6.9, 1000 15.1 / 11.3, 4000 32.3 / 30.2, but 12000 81 / 83
// (and width 2048, 4000 54.9 / 55.8: many tokens of many experts stay apart, ops.resadd_moe_router).
template <int NE, int XC>      // entries a thread, 8-wide chunks a lane
__global__ void __launch_bounds__(256) resadd_router_kernel(const u16* __restrict__ y, long ldy, const float* __restrict__ w, float* __restrict__ x,
                                                            u16* __restrict__ xl, int H, float eps, const float* __restrict__ bias,
                                                            const u16* __restrict__ wg, int E, int k, int* __restrict__ ids,
                                                            float* __restrict__ wts, int shared, float scale) {
  __shared__ float red[4], lgs[64];
  __shared__ __attribute__((aligned(16))) u16 rowb[512 * XC];
  const long row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nc = H >> 3;
  float* xr = x + row * (long)H;
  float a[NE], s[NE], g[NE], b[NE];
  const float* bp = bias ? bias : w;
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int c = min((int)threadIdx.x + 256 * j, H - 1);
    s[j] = xr[c];
    g[j] = w[c];
    a[j] = bf2f(y[row * ldy + c]);
    b[j] = bp[c];
  }
  uint4 wr[2][XC];
  auto rows = [&](int e0) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < XC; ++c) wr[i][c] = ld16(wg + (long)min(e0 + wave + 4 * i, E - 1) * H + 8 * min(lane + 64 * c, nc - 1));
  };
  rows(0);
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    if (bias) a[j] += b[j];
    const float v = (int)threadIdx.x + 256 * j < H ? a[j] : 0.f;
    q = fmaf(v, v, q);
  }
  q = wave_sum(q);
  if (lane == 0) red[wave] = q;
  __syncthreads();
  q = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) q += red[i];
  const float r = 1.f / sqrtf(q / (float)H + eps);
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int c = threadIdx.x + 256 * j;
    if (c >= H) continue;
    const float v = s[j] + a[j] * r * g[j];
    xr[c] = v;
    const u16 o = f2bf(v);
    xl[row * (long)H + c] = o;
    rowb[c] = o;
  }
  __syncthreads();
  uint4 xv[XC];
#pragma unroll
  for (int c = 0; c < XC; ++c) xv[c] = lane + 64 * c < nc ? ld16(rowb + 8 * (lane + 64 * c)) : make_uint4(0u, 0u, 0u, 0u);
  for (int e0 = 0; e0 < E; e0 += 8) {
    if (e0 > 0) rows(e0);
    float d[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      d[i] = 0.f;
#pragma unroll
      for (int c = 0; c < XC; ++c) {
        float f[8], h[8];
        unpack8(lane + 64 * c < nc ? wr[i][c] : make_uint4(0u, 0u, 0u, 0u), f);
        unpack8(xv[c], h);
#pragma unroll
        for (int u = 0; u < 8; ++u) d[i] += h[u] * f[u];
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1)
#pragma unroll
      for (int i = 0; i < 2; ++i) d[i] = lane_add(d[i], m);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (lane == 0 && e0 + wave + 4 * i < E) lgs[e0 + wave + 4 * i] = d[i];
  }
  __syncthreads();
  if (wave == 0) router_choice(lane < E ? lgs[lane] : -INFINITY, lane, E, k, row * (k + shared), ids, wts, shared, scale);
}

// buf = [n, idx0, val0, idx1, val1, ...]: dst[idx_i] = val_i.  n is read on the device, so a
// captured decode graph applies a different number of block-table updates on every replay.
__global__ void scatter_pairs_kernel(int* __restrict__ dst, const int* __restrict__ buf, int cap) {
  const int n = min(buf[0], cap);
  for (int i = threadIdx.x; i < n; i += blockDim.x) dst[buf[1 + 2 * i]] = buf[2 + 2 * i];
}
}  // namespace

// ---- decode-step I/O inside the step's graph (round 4).  The step's inputs are staged by the host
// in pinned, device-mapped memory and its sampled tokens are read back from pinned memory; moving
// them with these kernels instead of hipMemcpyAsync keeps every decode step ONE graph launch on
// one queue: an async H2D copy runs on an SDMA engine and waited ~320 us per step for the
// read-back blit of the previous step to signal it (profiles/r4_driver_window_gaps.md).
// step_fetch: dec_dev[0:n_dec] <- dec_host, except the input ids, which the pipelined decode takes
// from the previous step's sampled tokens still on the device: ids[i] = d_out[src[i]] where
// src[i] >= 0 (src lives in the host buffer at src_off); and the attention work list
// items_dev <- items_host, as many words as its header says (decode_work_items layout).
__global__ void __launch_bounds__(256) step_fetch_kernel(const int* __restrict__ dec_host, int* __restrict__ dec_dev,
                                                         int n_dec, int ids_off, int src_off, int n_ids,
                                                         const int* __restrict__ d_out,
                                                         const int* __restrict__ items_host,
                                                         int* __restrict__ items_dev, int items_cap,
                                                         int* __restrict__ sc_dst, int sc_off, int sc_cap) {
  const int stride = gridDim.x * blockDim.x;
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  int n_items = 0;
  if (items_host != nullptr) {
    const int h = items_host[0];
    n_items = min(h < 0 ? 4 + 4 * (-h) : 1 + 2 * h, items_cap);
  }
  for (int w = gid; w < n_dec; w += stride) {
    int v = dec_host[w];
    const int i = w - ids_off;
    if (i >= 0 && i < n_ids) {
      const int s = dec_host[src_off + i];
      if (s >= 0 && s < n_ids) v = d_out[s];
    }
    dec_dev[w] = v;
  }
  for (int w = gid; w < n_items; w += stride) items_dev[w] = items_host[w];
  if (sc_dst != nullptr)      // [n, idx0, val0, ...] of the host buffer: dst[idx] = val (a launch of its own: 2.5 to 4 us of a step)
    for (int i = gid; i < sc_cap; i += stride) {
      const int n = dec_host[sc_off], at = dec_host[sc_off + 1 + 2 * i], v = dec_host[sc_off + 2 + 2 * i];
      if (i < n) sc_dst[at] = v;
    }
}

// step_store: out_host[0:n] <- d_out (the sampled tokens, + the TP health vote), last node of the graph
__global__ void __launch_bounds__(256) step_store_kernel(const int* __restrict__ d_out, int* __restrict__ out_host,
                                                         int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out_host[i] = d_out[i];
}

static inline int grid_for(long n, int threads) {
  long g = (n + threads - 1) / threads;
  if (g > 65536) g = 65536;
  return g < 1 ? 1 : (int)g;
}

extern "C" int dllm_silu_mul(const void* gu, void* out, long T, int I, long in_stride, hipStream_t stream) {
  if (I % 8 != 0) return -1;
  const long n = T * (I / 8);
  if (n == 0) return 0;
  if (n >= (1L << 30)) return -2;
  hipLaunchKernelGGL(silu_mul_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, (const u16*)gu, (u16*)out, T, I,
                     in_stride);
  return (int)hipGetLastError();
}

extern "C" int dllm_embed(const int* ids, const void* table, void* out, long T, int H, long lo, long rows,
                          float* ssq, int* sc_dst, const int* sc_buf, int sc_cap, hipStream_t stream) {
  if (H % 8 != 0) return -1;
  if (T == 0 && sc_buf == nullptr) return 0;
  const unsigned grid = (unsigned)((T + 3) / 4) + (sc_buf != nullptr ? 1u : 0u);
  hipLaunchKernelGGL(embed_kernel, dim3(grid), dim3(256), 0, stream, ids, (const u16*)table, (u16*)out, T, H, lo, rows,
                     ssq, sc_dst, sc_buf, sc_cap);
  return (int)hipGetLastError();
}

extern "C" int dllm_gelu(const void* x, void* y, long n, hipStream_t stream) {
  if (n % 8 != 0) return -1;
  if (n == 0) return 0;
  hipLaunchKernelGGL(gelu_kernel, dim3(grid_for(n / 8, 256)), dim3(256), 0, stream, (const u16*)x, (u16*)y, n / 8);
  return (int)hipGetLastError();
}

// x [T, H] packed rows, 16-byte aligned, H % 8 == 0 and H <= 512
extern "C" int dllm_ln_pool_l2(const void* x, const void* w, const void* b, float eps, const int* lens, float* out, int B, int H, const int* starts,
                               int T, hipStream_t stream) {
  if (H < 8 || H % 8 || H > 512 || B < 1) return -1;
  hipLaunchKernelGGL(ln_pool_l2_kernel, dim3(B), dim3(512), 0, stream, (const u16*)x, (const u16*)w, (const u16*)b, eps, lens, out, H, starts, T);
  return (int)hipGetLastError();
}

extern "C" int dllm_mean_pool_l2(const void* x, const int* lens, float* out, int B, int S, int H, const int* starts, int T,
                                 hipStream_t stream) {
  if (H % 8 == 0 && H <= 2048 && ((uintptr_t)x & 15) == 0) {
    const size_t lds = (size_t)(256 / (H / 8)) * H * sizeof(float);      // at most 8 KB
    hipLaunchKernelGGL(mean_pool_l2_kernel, dim3(B), dim3(256), lds, stream, (const u16*)x, lens, out, S, H, starts, T);
    return (int)hipGetLastError();
  }
  int threads = ((H + 3) / 4 + 63) / 64 * 64;
  if (threads > 256 || threads * 4 < H) return -1;
  hipLaunchKernelGGL(mean_pool_any_kernel, dim3(B), dim3(threads), 0, stream, (const u16*)x, lens, out, S, H, starts, T);
  return (int)hipGetLastError();
}

extern "C" int dllm_scatter_pairs(int* dst, const int* buf, int cap, hipStream_t stream) {
  hipLaunchKernelGGL(scatter_pairs_kernel, dim3(1), dim3(256), 0, stream, dst, buf, cap);
  return (int)hipGetLastError();
}

extern "C" int dllm_moe_gate(const float* logits, int T, int E, int k, int* ids, float* w, hipStream_t stream) {
  if (E > 64 || k > 8 || k > E) return -1;
  if (T == 0) return 0;
  hipLaunchKernelGGL(moe_gate_kernel, dim3((T + 127) / 128), dim3(128), 0, stream, logits, T, E, k, ids, w);
  return (int)hipGetLastError();
}

extern "C" int dllm_moe_router(const void* x, long x_stride, const void* wg, int T, int E, int H, int k, int* ids,
                               float* w, float* logits, int shared, float scale, const void* norm_w, float eps, void* xn,
                               hipStream_t stream) {
  if (E > 64 || k > 8 || k > E || H % 8 != 0 || H > 8192 || x_stride % 8 != 0) return -1;
  if (T == 0) return 0;
  const dim3 grid((T + 3) / 4), block(256);
  const int nc = H / 8;
#define ROUTER(XC, EB)                                                                                                          \
  do {                                                                                                                          \
    if (norm_w)                                                                                                                 \
      hipLaunchKernelGGL((moe_router_kernel<XC, EB, true>), grid, block, 0, stream, (const u16*)x, x_stride, (const u16*)wg, T, E, H, k, \
                         ids, w, logits, shared, scale, (const u16*)norm_w, eps, (u16*)xn);                                     \
    else                                                                                                                        \
      hipLaunchKernelGGL((moe_router_kernel<XC, EB, false>), grid, block, 0, stream, (const u16*)x, x_stride, (const u16*)wg, T, E, H, k, \
                         ids, w, logits, shared, scale, nullptr, 0.f, nullptr);                                                 \
  } while (0)
  switch ((nc + 63) / 64) {      // (as many chunks a lane as the row has: none is loaded for nothing but in the last)
    case 1: ROUTER(1, 8); break;
    case 2: ROUTER(2, 8); break;
    case 3: ROUTER(3, 4); break;
    case 4: ROUTER(4, 4); break;
    case 5: ROUTER(5, 2); break;
    case 6: ROUTER(6, 2); break;
    case 7: case 8: ROUTER(8, 2); break;
    case 9: case 10: case 11: case 12: ROUTER(12, 2); break;
    default: ROUTER(16, 2);
  }
#undef ROUTER
  return (int)hipGetLastError();
}

// y [T, H] bf16 rows, x [T, H] f32 in place, xl [T, H] bf16; wg [E, H] bf16, rows of 16 bytes; ids and wts [T, k + shared]
extern "C" int dllm_resadd_router(const void* y, long ldy, const float* w, float eps, float* x, void* xl, const float* bias, const void* wg, int T,
                                  int E, int H, int k, int* ids, float* wts, int shared, float scale, hipStream_t stream) {
  if (E < 1 || E > 64 || k < 1 || k > 8 || k > E || H < 8 || H % 8 || H > 2048) return -1;
  if (T == 0) return 0;
#define RR(NE, XC)                                                                                                                         \
  hipLaunchKernelGGL((resadd_router_kernel<NE, XC>), dim3(T), dim3(256), 0, stream, (const u16*)y, ldy, w, x, (u16*)xl, H, eps, bias, (const u16*)wg, \
                     E, k, ids, wts, shared, scale)
  if (H <= 512) RR(2, 1); else if (H <= 1024) RR(4, 2); else RR(8, 4);
#undef RR
  return (int)hipGetLastError();
}

extern "C" int dllm_step_fetch(const int* dec_host, int* dec_dev, int n_dec, int ids_off, int src_off, int n_ids,
                               const int* d_out, const int* items_host, int* items_dev, int items_cap, int* sc_dst, int sc_off,
                               int sc_cap, hipStream_t stream) {
  if (sc_dst != nullptr && (sc_off < 0 || sc_cap < 0 || sc_off + 1 + 2 * (long)sc_cap > n_dec)) return -3;
  if (n_dec <= 0 || ids_off < 0 || src_off < 0 || ids_off + n_ids > n_dec || src_off + n_ids > n_dec) return -1;
  if ((items_host == nullptr) != (items_dev == nullptr)) return -2;
  hipLaunchKernelGGL(step_fetch_kernel, dim3(32), dim3(256), 0, stream, dec_host, dec_dev, n_dec, ids_off, src_off,
                     n_ids, d_out, items_host, items_dev, items_cap, sc_dst, sc_off, sc_cap);
  return (int)hipGetLastError();
}

extern "C" int dllm_step_store(const int* d_out, int* out_host, int n, hipStream_t stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(step_store_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, d_out, out_host, n);
  return (int)hipGetLastError();
}
