// Grouped-query softmax attention over paged keys / values with any head widths (gfx950, wave64).
//
//   attn_prep   one workgroup per token: rotate-half positions on the first `rot` dims of every q / k
//               head, each head to unit RMS (f32), q times a per-head scale; k and v go to their
//               page slots, q to a dense [T, H, d] buffer.
//   qk_norm_prep  attention inputs with biases, a weighted RMS norm of every q / k vector before its
//               rotation, and `maps` score maps per head (differential attention: 2): query rows of
//               one key/value head leave ordered (map, head in group), so the grouped-query kernels
//               below pair them with key head (kv head, map); diff_combine merges the two maps.
//   proj_norm_prep  attention inputs whose q / k RMS norm runs over the whole projection (all heads
//               together, weights of that length) before the rotation; rotary pairs (2i, 2i + 1) or
//               (i, i + rot / 2); a per-head q scale; optionally every value head to unit RMS.
//   paged_gqa   one workgroup per (tile of new tokens, key/value head, group of <= 16 query heads):
//               its rows are tokens x query heads of the group (<= 16).  Keys are walked in tiles
//               staged in LDS as f32; a lane owns a key for the scores (one K read feeds the wave's
//               four rows), f32 online softmax per row, then a lane owns value dims for the weighted
//               sum (one V read feeds four rows).  The output is multiplied by sigmoid(gate).
//
//   gqa_f32     the f32 form on the f32 matrix cores: a wave per 16-key page, no LDS until the waves of a
//               workgroup meet (whole pages of 16 keys, widths up to 128, a value head per key head; paged_gqa takes the rest).
//
//   paged_gqa_mfma  the bf16 form on the matrix cores: 64 rows per workgroup, 16 per wave, so a row's
//               softmax never leaves its wave.  Q stays in registers as MFMA operands; a 64-key tile is
//               staged once for the four waves (K row-major, V already transposed in its page);
//               scores on v_mfma_f32_16x16x32_bf16 with f32 sums; online softmax in the accumulator
//               layout (row maxima over the 16 lanes of a DPP row); the weights go through the wave's
//               own LDS patch as bf16 hi + lo parts, so the weighted sum sees them to 16 bits of
//               mantissa through two MFMAs.  Key blocks above a wave's newest row are skipped.
//
//   rope_prep   attention inputs without a q / k norm: optional biases, rotate-half positions on the first
//               `rot` dims, q times one scale and optionally a number of its position; the launch also squares
//               the relu of a feed-forward's up columns that the same projection made (latent_prep: the
//               same beside a normed latent).
//
// Both attention kernels take a window (a row at position p sees keys p - win < j <= p) or a chunk (it
// sees the keys of its own chunk of positions, [p - p % chunk, p]), kept first keys (j < keep stays
// visible at any distance; the tiles between the kept keys and the window are not read), a soft cap on
// the scores (cap tanh(s / cap)) and a sink: one more term of the denominator, with no value, either
// exp(0) times `sink` or exp(sinks[head]).  Under a cap the matrix-core form keeps no running maximum.
// slopes: a head's scores fall by slopes[head] per position between row and key (not beside a cap); the
// matrix-core form starts its score accumulators there.  The gate has one logit per output entry or
// (ghead) one per head.
//
// Cache layout: K [blocks, G, block, d], V [blocks, G, dv, block] (bf16 or f32 like the activations;
// V is kept transposed inside its page because the weighted sum runs over keys); every score,
// weight and sum is f32.
#include "common.h"

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <typename T> __device__ __forceinline__ void stf(T* p, float v);
template <> __device__ __forceinline__ void stf<u16>(u16* p, float v) { *p = f2bf(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }

// The oldest key a row at position p sees (kept first keys apart): its window's, its chunk's, or 0.
__device__ __forceinline__ int oldest_key(int p, int win, int chunk) {
  return chunk > 0 ? p - p % chunk : (win > 0 ? max(0, p - win + 1) : 0);
}
// cap tanh(s / cap) = cap - 2 cap / (exp(2 s / cap) + 1); an overflowing exponential gives cap
__device__ __forceinline__ float cap_fast(float s, float cap, float two_over_cap) {
  return cap - 2.f * cap * __builtin_amdgcn_rcpf(__expf(s * two_over_cap) + 1.f);
}

// this workgroup's share of a token's row of a [T, zw] buffer of 4-byte words, cleared: the attention output of a step with padding rows,
// which no attention tile writes (a fill of its own: 4.7 us a layer of a decode step)
__device__ __forceinline__ void clear_row(uint32_t* zrow, int zw, long tok) {
  if (zrow)
    for (int i = blockIdx.y * 256 + threadIdx.x; i < zw; i += gridDim.y * 256) zrow[tok * zw + i] = 0u;
}

template <typename T>
__global__ void __launch_bounds__(256) attn_prep_kernel(const T* __restrict__ proj, long ld, int H, int G, int d, int dv,
                                                        const float* __restrict__ cos_sin, int tab_w, int rot, float eps,
                                                        const float* __restrict__ qscale, const int* __restrict__ pos,
                                                        const int* __restrict__ slots, T* __restrict__ kc,
                                                        T* __restrict__ vc, T* __restrict__ q, int BSZ, uint32_t* __restrict__ zrow,
                                                        int zw) {
  const long tok = blockIdx.x;
  clear_row(zrow, zw, tok);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const T* r = proj + tok * ld;
  const int slot = slots[tok];
  const long blk = slot >= 0 ? slot / BSZ : 0;
  const int off = slot >= 0 ? slot % BSZ : 0;
  const int half = rot >> 1;
  const float* cs = cos_sin + (long)pos[tok] * tab_w;
  const int hh = blockIdx.y * 4 + wave;     // q heads, then k heads, are consecutive in the projection
  if (hh < H + G && (hh < H || slot >= 0)) {
    const bool is_q = hh < H;
    const T* x = r + (long)hh * d;
    float ss = 0.f;
    for (int i = lane; i < d; i += 64) {
      float v = ldf(x + i);
      if (i < rot) {
        const int f = i < half ? i : i - half;
        const float c = cs[f], sn = cs[half + f];
        const float p = ldf(x + (i < half ? i + half : i - half));
        v = i < half ? v * c - p * sn : v * c + p * sn;
      }
      ss += v * v;
    }
    ss = wave_sum(ss);
    const float sc = (is_q ? qscale[hh] : 1.f) / sqrtf(ss / (float)d + eps);
    T* dst = is_q ? q + (tok * H + hh) * d : kc + ((blk * G + (hh - H)) * BSZ + off) * d;
    for (int i = lane; i < d; i += 64) {
      float v = ldf(x + i);
      if (i < rot) {
        const int f = i < half ? i : i - half;
        const float c = cs[f], sn = cs[half + f];
        const float p = ldf(x + (i < half ? i + half : i - half));
        v = i < half ? v * c - p * sn : v * c + p * sn;
      }
      stf(dst + i, v * sc);
    }
  }
  if (slot >= 0) {   // values: this workgroup's share of the G * dv entries
    const T* v = r + (long)(H + G) * d;
    for (int i = blockIdx.y * 256 + threadIdx.x; i < G * dv; i += gridDim.y * 256)
      vc[((blk * G + i / dv) * dv + i % dv) * BSZ + off] = v[i];
  }
}

// The same in 16-byte vectors (bf16): D / 8 lanes a head, a wave 512 / D heads of a token and four tokens with every load in flight; a
// workgroup covers 16 tokens (blockIdx.x) and one such group of heads, or (the last blockIdx.y) 512 value entries, turned in LDS so that
// the 16 tokens of an entry, which lie side by side in V^T's page, are stored by neighbouring lanes.  Element by element it is bound by
// 2-byte accesses, made twice, and by a sector for each value: 7300 tokens, 32 + 8 heads of 64 and as many values 123 us, here 32 (the
// bytes alone: 15).  Where it begins: dllm_attn_prep.
// A lane's eight squares are added in the order that the wave's exchanges have there (D = 64: the same bits).
constexpr int APV_T = 16, APV_V = 512;
template <int D>
__global__ void __launch_bounds__(256) attn_prep_vec_kernel(const u16* __restrict__ proj, long ld, int H, int G, int dv,
                                                            const float* __restrict__ cos_sin, int tab_w, int rot, float eps,
                                                            const float* __restrict__ qscale, const int* __restrict__ pos,
                                                            const int* __restrict__ slots, u16* __restrict__ kc, u16* __restrict__ vc,
                                                            u16* __restrict__ q, int BSZ, int T, int ny,
                                                            uint32_t* __restrict__ zrow, int zw) {
  constexpr int LPH = D / 8, TW = APV_T / 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t0 = blockIdx.x * APV_T;
  for (int t = t0; t < min(t0 + APV_T, T); ++t) clear_row(zrow, zw, t);
  if ((int)blockIdx.y < ny) {
    const int hh = (blockIdx.y * 64 + lane) / LPH, c = lane % LPH * 8, half = rot >> 1;
    const int hx = min(hh, H + G - 1), f = c < half ? c : c - half;
    const bool is_q = hh < H, turn = c < rot;
    const float qs = qscale[min(hh, H - 1)];
    uint4 x[TW], p[TW];
    f32x4 cs[TW][2], sn[TW][2];
    int slot[TW];
#pragma unroll
    for (int k = 0; k < TW; ++k) {
      const int tok = min(t0 + wave + 4 * k, T - 1);
      const u16* r = proj + tok * ld + hx * D;
      x[k] = ld16(r + c);
      slot[k] = slots[tok];
      if (turn) {
        p[k] = ld16(r + (c < half ? c + half : c - half));
        const float* cp = cos_sin + (long)pos[tok] * tab_w + f;
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          cs[k][y] = *reinterpret_cast<const f32x4*>(cp + 4 * y);
          sn[k][y] = *reinterpret_cast<const f32x4*>(cp + half + 4 * y);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < TW; ++k) {
      const int tok = t0 + wave + 4 * k;
      float v[8], w[8], e[8];
      unpack8(x[k], v);
      if (turn) {
        unpack8(p[k], w);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float co = cs[k][j / 4][j % 4], si = sn[k][j / 4][j % 4];
          v[j] = c < half ? v[j] * co - w[j] * si : v[j] * co + w[j] * si;
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = v[j] * v[j];
#pragma unroll
      for (int o = LPH / 2; o > 0; o >>= 1)
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = lane_add(e[j], o);
      const float ss = ((e[0] + e[4]) + (e[2] + e[6])) + ((e[1] + e[5]) + (e[3] + e[7]));
      const float sc = (is_q ? qs : 1.f) / sqrtf(ss / (float)D + eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] *= sc;
      if (tok >= T || hh >= H + G || (!is_q && slot[k] < 0)) continue;
      u16* dst = is_q ? q + ((long)tok * H + hh) * D : kc + (((long)(slot[k] / BSZ) * G + (hh - H)) * BSZ + slot[k] % BSZ) * D;
      st16(dst + c, pack8(v));
    }
    return;
  }
  __shared__ __attribute__((aligned(16))) u16 sv[APV_T][APV_V + 8];
  const int e0 = (blockIdx.y - ny) * APV_V, ne = min(APV_V, G * dv - e0);      // whole vectors of 8
  for (int i = threadIdx.x; i < APV_T * (APV_V / 8); i += 256) {
    const int t = i / (APV_V / 8), c = i % (APV_V / 8) * 8;
    if (t0 + t < T && c < ne) st16(&sv[t][c], ld16(proj + (t0 + t) * ld + (long)(H + G) * D + e0 + c));
  }
  const int t = lane % APV_T, slot = t0 + t < T ? slots[t0 + t] : -1;
  __syncthreads();
  if (slot < 0) return;
  const long blk = slot / BSZ;
  u16* vp = vc + blk * G * dv * BSZ + slot % BSZ;
  for (int i = threadIdx.x / APV_T; i < ne; i += 256 / APV_T) vp[(long)(e0 + i) * BSZ] = sv[t][i];
}

// One wave per q / k vector (head, map): bias, weighted RMS norm over d, rotate-half positions on the
// first `rot` dims, q times `qscale`.  Query unit (h, m) of key/value head g = h / R leaves as row
// g M R + m R + h % R of q [T, H M, d]; key unit (g, m) goes to key head g M + m of the page.
template <typename T>
__global__ void __launch_bounds__(256) qk_norm_prep_kernel(const T* __restrict__ proj, long ld, const float* __restrict__ bias,
                                                           int H, int G, int M, int d, int dv,
                                                           const float* __restrict__ qw, const float* __restrict__ kw,
                                                           const float* __restrict__ cos_sin, int tab_w, int rot, float eps,
                                                           float qscale, const int* __restrict__ pos,
                                                           const int* __restrict__ slots, T* __restrict__ kc,
                                                           T* __restrict__ vc, T* __restrict__ q, int BSZ,
                                                           uint32_t* __restrict__ zrow, int zw) {
  const long tok = blockIdx.x;
  clear_row(zrow, zw, tok);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;      // (a scalar number here cost 3000 tokens 15 %)
  const T* r = proj + tok * ld;
  const int slot = kc ? slots[tok] : -1;
  const long blk = slot >= 0 ? slot / BSZ : 0;
  const int off = slot >= 0 ? slot % BSZ : 0;
  const int half = rot >> 1;
  const float* cs = cos_sin + (long)pos[tok] * tab_w;
  const int nq = H * M, nk = kc ? G * M : 0;
  const int u = blockIdx.y * 4 + wave;     // q units, then k units, are consecutive in the projection
  if (u < nq + nk && (u < nq || slot >= 0)) {
    const bool is_q = u < nq;
    const T* x = r + (long)u * d;
    const float* b = bias ? bias + (long)u * d : nullptr;
    const float* w = is_q ? qw : kw;
    float ss = 0.f;
    for (int i = lane; i < d; i += 64) {
      const float v = ldf(x + i) + (b ? b[i] : 0.f);
      ss += v * v;
    }
    const float sc = 1.f / sqrtf(wave_sum(ss) / (float)d + eps);
    T* dst;
    if (is_q) {
      const int h = u / M, m = u % M, R = H / G;
      dst = q + (tok * nq + (long)(h / R) * M * R + m * R + h % R) * d;
    } else {
      dst = kc + ((blk * nk + (u - nq)) * BSZ + off) * d;
    }
    const float os = is_q ? qscale : 1.f;
    for (int i = lane; i < d; i += 64) {
      float v = (ldf(x + i) + (b ? b[i] : 0.f)) * sc * w[i];
      if (i < rot) {
        const int f = i < half ? i : i - half;
        const int j = i < half ? i + half : i - half;
        const float c = cs[f], sn = cs[half + f];
        const float p = (ldf(x + j) + (b ? b[j] : 0.f)) * sc * w[j];
        v = i < half ? v * c - p * sn : v * c + p * sn;
      }
      stf(dst + i, v * os);
    }
  }
  if (slot >= 0) {   // values: this workgroup's share of the G * dv entries
    const long vo = (long)(nq + nk) * d;
    for (int i = blockIdx.y * 256 + threadIdx.x; i < G * dv; i += gridDim.y * 256)
      stf(vc + ((blk * G + i / dv) * dv + i % dv) * BSZ + off, ldf(r + vo + i) + (bias ? bias[vo + i] : 0.f));
  }
}

// One workgroup per token.  q (H d entries) and k (G d entries) are each normed over their whole
// length with weights qw / kw, then rotated on the first `rot` dims of every head: pairs (2i, 2i + 1)
// when `inter`, else (i, i + rot / 2), angle index i; q times qscale[head].  vnorm: every value head
// divided by its root mean square.  kc null: proj holds q alone.
template <typename T>
__global__ void __launch_bounds__(256) proj_norm_prep_kernel(const T* __restrict__ proj, long ld, int H, int G, int d, int dv,
                                                             const float* __restrict__ qw, const float* __restrict__ kw,
                                                             const float* __restrict__ cos_sin, int tab_w, int rot,
                                                             int inter, float eps, const float* __restrict__ qscale,
                                                             int vnorm, const int* __restrict__ pos,
                                                             const int* __restrict__ slots, T* __restrict__ kc,
                                                             T* __restrict__ vc, T* __restrict__ q, int BSZ,
                                                             T* __restrict__ zrow, int zn) {
  // zrow: a [T, zn] buffer whose row of this token is cleared (the attention output of a step with
  // padding rows, which no attention tile writes)
  __shared__ float red[16];
  const long tok = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (zrow)
    for (int e = tid; e < zn; e += 256) stf(zrow + tok * zn + e, 0.f);
  const T* r = proj + tok * ld;
  const int slot = kc ? slots[tok] : -1;
  const long blk = slot >= 0 ? slot / BSZ : 0;
  const int off = slot >= 0 ? slot % BSZ : 0;
  const int half = rot >> 1;
  const float* cs = cos_sin + (long)pos[tok] * tab_w;
  const int nq = H * d, nk = slot >= 0 ? G * d : 0;
  float sq = 0.f, sk = 0.f;
  for (int e = tid; e < nq; e += 256) { const float v = ldf(r + e); sq += v * v; }
  for (int e = tid; e < nk; e += 256) { const float v = ldf(r + nq + e); sk += v * v; }
  const float rq = 1.f / sqrtf(block_sum(sq, red) / (float)nq + eps);
  const float rk = nk ? 1.f / sqrtf(block_sum(sk, red) / (float)nk + eps) : 0.f;   // slot is uniform in the workgroup
  // a wave per q / k head, a lane per dim: no index arithmetic beyond adds
  const int units = H + (nk ? G : 0);
  for (int un = wave; un < units; un += 4) {
    const bool is_q = un < H;
    const int hh = is_q ? un : un - H;
    const T* x = r + (is_q ? 0 : nq) + hh * d;              // this head's columns
    const float* w = (is_q ? qw : kw) + hh * d;
    const float sc = is_q ? rq : rk;
    const float os = is_q ? qscale[hh] : 1.f;
    T* dst = is_q ? q + (tok * H + hh) * d : kc + ((blk * G + hh) * BSZ + off) * d;
    for (int i = lane; i < d; i += 64) {
      float v = ldf(x + i) * sc * w[i];
      if (i < rot) {
        int j, f;
        bool first;
        if (inter) { j = i ^ 1; f = i >> 1; first = !(i & 1); }
        else { first = i < half; j = first ? i + half : i - half; f = first ? i : i - half; }
        const float cc = cs[f], sn = cs[half + f];
        const float pv = ldf(x + j) * sc * w[j];
        v = first ? v * cc - pv * sn : v * cc + pv * sn;
      }
      stf(dst + i, v * os);
    }
  }
  if (slot >= 0) {   // values: a wave per value head
    const T* vv = r + nq + nk;
    for (int g = wave; g < G; g += 4) {
      float sv = 1.f;
      if (vnorm) {
        float ss = 0.f;
        for (int i = lane; i < dv; i += 64) { const float v = ldf(vv + g * dv + i); ss += v * v; }
        sv = 1.f / sqrtf(wave_sum(ss) / (float)dv + eps);
      }
      for (int i = lane; i < dv; i += 64) stf(vc + ((blk * G + g) * dv + i) * BSZ + off, ldf(vv + g * dv + i) * sv);
    }
  }
}

// Squared relu of a row's up columns (this workgroup's share): act[i] = relu(up[i])^2.  vec: rows of whole
// 16-byte vectors on both sides.
template <typename T>
__device__ __forceinline__ void act_share(const T* __restrict__ up, int ff, T* __restrict__ act, int part, int parts, int tid,
                                          bool vec) {
  for (int i = part * 256 + tid; i < ff; i += parts * 256) {
    const float v = fmaxf(ldf(up + i), 0.f);
    stf(act + i, v * v);
  }
}
template <>
__device__ __forceinline__ void act_share<u16>(const u16* __restrict__ up, int ff, u16* __restrict__ act, int part, int parts,
                                               int tid, bool vec) {
  if (vec) {
    for (int i = 8 * (part * 256 + tid); i < ff; i += 8 * parts * 256) {
      float f[8];
      unpack8(ld16(up + i), f);
#pragma unroll
      for (int x = 0; x < 8; ++x) { f[x] = fmaxf(f[x], 0.f); f[x] *= f[x]; }
      st16(act + i, pack8(f));
    }
    return;
  }
  for (int i = part * 256 + tid; i < ff; i += parts * 256) {
    const float v = fmaxf(bf2f(up[i]), 0.f);
    act[i] = f2bf(v * v);
  }
}

// Attention inputs without a q / k norm, and the activation of a feed-forward that shares the
// projection.  proj row: q (H d) | k (G d) | v (G dv) | ...; a wave per q / k head: rotate-half
// positions on the first `rot` dims (cos and sin as the table holds them), q times qscale; k and v to
// their page slots.  act (null: no feed-forward): act[tok] = relu(proj[tok, ucol : ucol + ff])^2.
// zrow: the first zn columns of a padding token's row (slot < 0) are cleared (an attention output whose
// padding rows no tile writes).  bias (f32 over the q | k | v columns) is added before the rotation; qtab:
// q is also multiplied by qtab[position].
template <typename T>
__global__ void __launch_bounds__(256) rope_prep_kernel(const T* __restrict__ proj, long ld, int H, int G, int d, int dv,
                                                        const float* __restrict__ cos_sin, int tab_w, int rot, float qscale,
                                                        const int* __restrict__ pos, const int* __restrict__ slots,
                                                        T* __restrict__ kc, T* __restrict__ vc, T* __restrict__ q, int BSZ,
                                                        int ucol, int ff, T* __restrict__ act, long lda, int vec,
                                                        T* __restrict__ zrow, long ldz, int zn, const float* __restrict__ bias,
                                                        const float* __restrict__ qtab) {
  const long tok = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* r = proj + tok * ld;
  const int slot = slots[tok];
  const long blk = slot >= 0 ? slot / BSZ : 0;
  const int off = slot >= 0 ? slot % BSZ : 0;
  const int half = rot >> 1;
  const float* cs = cos_sin + (long)pos[tok] * tab_w;
  if (zrow && slot < 0)
    for (int i = blockIdx.y * 256 + tid; i < zn; i += gridDim.y * 256) stf(zrow + tok * ldz + i, 0.f);
  for (int hh = blockIdx.y * 4 + wave; hh < H + G; hh += gridDim.y * 4) {   // q heads, then k heads
    const bool is_q = hh < H;
    if (!is_q && slot < 0) continue;
    const T* x = r + (long)hh * d;
    const float* b = bias ? bias + (long)hh * d : nullptr;
    T* dst = is_q ? q + (tok * H + hh) * d : kc + ((blk * G + (hh - H)) * BSZ + off) * d;
    const float os = is_q ? (qtab ? qscale * qtab[pos[tok]] : qscale) : 1.f;
    for (int i = lane; i < d; i += 64) {
      float v = ldf(x + i) + (b ? b[i] : 0.f);
      if (i < rot) {
        const bool first = i < half;
        const int f = first ? i : i - half, j = first ? i + half : i - half;
        const float c = cs[f], sn = cs[half + f];
        const float p = ldf(x + j) + (b ? b[j] : 0.f);
        v = first ? v * c - p * sn : v * c + p * sn;
      }
      stf(dst + i, v * os);
    }
  }
  if (slot >= 0) {   // values: this workgroup's share of the G * dv entries
    const T* v = r + (long)(H + G) * d;
    const float* b = bias ? bias + (long)(H + G) * d : nullptr;
    for (int i = blockIdx.y * 256 + tid; i < G * dv; i += gridDim.y * 256) {
      T* dst = vc + ((blk * G + i / dv) * dv + i % dv) * BSZ + off;
      if (b) stf(dst, ldf(v + i) + b[i]);
      else *dst = v[i];
    }
  }
  if (act) act_share<T>(r + ucol, ff, act + tok * lda, blockIdx.y, gridDim.y, tid, vec);
}

// a [T, G, 2, R, dv] f32 (the two maps' outputs) -> out [T, G R, dv] = unit-RMS(a1 - lam a2) * scale:
// one wave per (token, head)
template <typename T>
__global__ void __launch_bounds__(256) diff_combine_kernel(const float* __restrict__ a, T* __restrict__ out, long units, int H,
                                                           int G, int dv, float lam, float eps, float scale) {
  const long u = (long)blockIdx.x * 4 + (threadIdx.x >> 6);      // (in a scalar: its divisions took 4000 rows of 16 heads of 64 from 20.9 to 23.3 us)
  const int lane = threadIdx.x & 63;
  if (u >= units) return;
  const long tok = u / H;
  const int h = (int)(u % H), R = H / G;
  const float* a1 = a + ((tok * G + h / R) * 2 * R + h % R) * dv;
  const float* a2 = a1 + (long)R * dv;
  float ss = 0.f;
  for (int i = lane; i < dv; i += 64) {
    const float o = a1[i] - lam * a2[i];
    ss += o * o;
  }
  const float sc = scale / sqrtf(wave_sum(ss) / (float)dv + eps);
  for (int i = lane; i < dv; i += 64) stf(out + u * dv + i, (a1[i] - lam * a2[i]) * sc);
}

constexpr int GA_ROWS = 16;   // rows per workgroup
// up to a workgroup per CU, 8 waves share a workgroup's keys, past that 4 (16 heads of 64, us with 8 / 4: 128 workgroups of 400
// keys 11.9 / 14.8, 8 of 2000 34 / 49, 480 of 60 9.9 / 6.8, 2016 of up to 200 62 / 39; 16 waves, without registers for a page ahead: 8 of 400
// keys 11.4 against 10.9, of 2000 31 against 34)
constexpr int GQF_WIDE = 256;

// KT keys per tile (64, or 32 when the tile would not fit the LDS), NJ = ceil(dv / 64)
template <typename T, int NJ>
__global__ void __launch_bounds__(256) paged_gqa_kernel(const T* __restrict__ q, const T* __restrict__ kc,
                                                        const T* __restrict__ vc, const int* __restrict__ bt, int bt_ld,
                                                        int BSZ, const int* __restrict__ qstart,
                                                        const int* __restrict__ qlen, const int* __restrict__ ctx,
                                                        const int* __restrict__ tile_seq, const int* __restrict__ tile_tok0,
                                                        const T* __restrict__ gate, long ldg, T* __restrict__ out, int H,
                                                        int G, int d, int dv, int TQ, int KT, int win, int GV,
                                                        float* __restrict__ out32, int keep, float sink, int chunk,
                                                        float cap, const float* __restrict__ sinks, long ldo,
                                                        const float* __restrict__ slopes, int ghead) {
  // win > 0: a row at position p sees keys p - win < j <= p, and keys j < keep; chunk > 0: keys of its
  // own chunk.  GV value heads: key head g reads value head g / (G / GV).  out32: the output stays f32.
  // sink: one more term of score 0 and that weight in the denominator; sinks: of score sinks[head].
  extern __shared__ float sm[];
  const int s = tile_seq[blockIdx.x];
  const int n = qlen[s];
  const int tok0 = tile_tok0[blockIdx.x];
  if (n <= 0 || tok0 >= n) return;   // the whole workgroup (padding tiles)
  const int g = blockIdx.y, R = H / G;
  const int r0 = blockIdx.z * GA_ROWS, Rh = min(GA_ROWS, R - r0);
  const int nq = min(TQ, n - tok0), nrows = nq * Rh;
  const int q0 = qstart[s], p0 = ctx[s] - n;
  const int dp = d | 1;
  float* Qs = sm;                      // [16][d]
  float* Ks = Qs + GA_ROWS * d;        // [KT][d | 1]
  float* Vs = Ks + KT * dp;            // [KT][dv]
  float* Ps = Vs + KT * dv;            // [16][64]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // row rr -> (token tok0 + rr / Rh, query head g R + r0 + rr % Rh); rows past nrows are idle
  for (int e = tid; e < GA_ROWS * d; e += 256) {
    const int rr = e / d, i = e % d;
    float v = 0.f;
    if (rr < nrows) v = ldf(q + ((long)(q0 + tok0 + rr / Rh) * H + g * R + r0 + rr % Rh) * d + i);
    Qs[e] = v;
  }
  float m[4], l[4], O[4][NJ], slp[4];
  int rpos[4], rlo[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int rr = wave + 4 * x;
    m[x] = -INFINITY;
    l[x] = 0.f;
    rpos[x] = rr < nrows ? p0 + tok0 + rr / Rh : -1;   // -1: sees no key
    rlo[x] = rr < nrows ? oldest_key(rpos[x], win, chunk) : 0;
    slp[x] = slopes && rr < nrows ? slopes[g * R + r0 + rr % Rh] : 0.f;
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) O[x][jj] = 0.f;
  }
  const int last = p0 + tok0 + nq - 1;   // the newest key any row sees
  const int* btr = bt + (long)s * bt_ld;
  const int gv = g / (G / GV);
  const int first = oldest_key(p0 + tok0, win, chunk);   // the oldest key any row sees
  for (int k0 = (keep > 0 ? 0 : first / KT * KT); k0 <= last; k0 += KT) {
    if (k0 >= keep && k0 + KT <= first) continue;   // between the kept keys and the window (uniform in the workgroup)
    const int nk = min(KT, last + 1 - k0);
    __syncthreads();   // the previous tile is consumed (and Qs is written)
    for (int e = tid; e < KT * d; e += 256) {
      const int kk = e / d, i = e % d;
      float v = 0.f;
      if (kk < nk) {
        const int pk = k0 + kk;
        v = ldf(kc + (((long)btr[pk / BSZ] * G + g) * BSZ + pk % BSZ) * d + i);
      }
      Ks[kk * dp + i] = v;
    }
    for (int e = tid; e < KT * dv; e += 256) {
      const int kk = e / dv, jx = e % dv;
      float v = 0.f;
      if (kk < nk) {
        const int pk = k0 + kk;
        v = ldf(vc + (((long)btr[pk / BSZ] * GV + gv) * dv + jx) * BSZ + pk % BSZ);
      }
      Vs[e] = v;
    }
    __syncthreads();
    // scores: lane = key; the wave's rows are wave, wave + 4, wave + 8, wave + 12
    float sc[4] = {0.f, 0.f, 0.f, 0.f};
    if (lane < KT) {
      const float* kr = Ks + lane * dp;
#pragma unroll 4
      for (int i = 0; i < d; ++i) {
        const float kv = kr[i];
#pragma unroll
        for (int x = 0; x < 4; ++x) sc[x] += Qs[(wave + 4 * x) * d + i] * kv;
      }
    }
    const int pk = k0 + lane;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const bool vis = lane < nk && pk <= rpos[x] && (pk >= rlo[x] || pk < keep);
      const float sv = !vis ? -INFINITY : cap > 0.f ? cap * tanhf(sc[x] / cap) : slopes ? sc[x] - slp[x] * (float)(rpos[x] - pk) : sc[x];
      const float mn = fmaxf(m[x], wave_max(sv));
      float p = 0.f, f = 1.f;
      if (mn > -INFINITY) {
        p = vis ? expf(sv - mn) : 0.f;
        f = expf(m[x] - mn);    // m = -inf before the first visible key: f = 0, and O and l are 0
      }
      l[x] = l[x] * f + wave_sum(p);
      m[x] = mn;
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) O[x][jj] *= f;
      Ps[(wave + 4 * x) * 64 + lane] = p;
    }
    __syncthreads();
    // weighted sum: lane owns value dims lane, lane + 64, ...
    for (int kk = 0; kk < nk; ++kk) {
      float vv[NJ];
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) vv[jj] = lane + 64 * jj < dv ? Vs[kk * dv + lane + 64 * jj] : 0.f;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float p = Ps[(wave + 4 * x) * 64 + kk];
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) O[x][jj] += p * vv[jj];
      }
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int rr = wave + 4 * x;
    if (rr >= nrows) continue;
    const long tok = q0 + tok0 + rr / Rh;
    const int h = g * R + r0 + rr % Rh;
    const float inv = 1.f / (l[x] + (sinks ? expf(sinks[h] - m[x]) : sink > 0.f ? sink * expf(-m[x]) : 0.f));
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
      const int jx = lane + 64 * jj;
      if (jx >= dv) continue;
      float o = O[x][jj] * inv;
      if (gate) o *= 1.f / (1.f + expf(-ldf(gate + tok * ldg + (ghead ? (long)h : (long)h * dv + jx))));
      if (out32) out32[tok * ldo + (long)h * dv + jx] = o;
      else stf(out + tok * ldo + (long)h * dv + jx, o);
    }
  }
}

// ---------------------------------------------------------------- f32 on the matrix cores
// A wave takes a 16-key page at a time, alone: S^T = K Q^T (keys 4 g4 + i of a lane against row lr), so that a row's softmax
// is four registers and two lane exchanges, and its weights are at once the right operand of O^T = V^T P^T.  Every operand
// comes from where it lies, 16 bytes a lane (contraction step x of lane group g4 stands for dim 16 b + 4 g4 + x, or key
// 4 g4 + x): no LDS and no barrier until the NW waves of a workgroup, which take every NW-th page, meet at the end.  The next
// page's keys and values travel while one is computed.  Bounded by one page's load and 32 small products at decode, by the
// f32 matrix rate (139 TF/s) over prompts.  At the end every wave leaves its sums in LDS and a thread an output adds them up, in the order of the
// waves; its gate is asked for at the start.  (Halves of the waves adding to the other halves, two barriers each, and a last wave that then
// read the gates of all rows were 4 us of any launch.)  16 query heads of 64 on 4 key heads: two sequences of 400 keys 11.0 us a step (14.8
// with that end; 104 in the general kernel above), one of 60 5.6 (9.1), a prompt of 2000 tokens 138 (144; 1087); heads of 128, two of 400 keys
// 19 (26).  Errors against 64 bits 2e-7 either way.
template <int KB, int VB, int NW>
__global__ void __launch_bounds__(64 * NW) gqa_f32_kernel(const float* __restrict__ q, const float* __restrict__ kc,
                                                          const float* __restrict__ vc, const int* __restrict__ bt, int bt_ld,
                                                          int BSZ, const int* __restrict__ qstart, const int* __restrict__ qlen,
                                                          const int* __restrict__ ctx, const int* __restrict__ tile_seq,
                                                          const int* __restrict__ tile_tok0, const float* __restrict__ gate,
                                                          long ldg, float* __restrict__ out, int H, int G, int d, int dv, int TQ,
                                                          int win, int keep, float sink, int chunk, float cap,
                                                          const float* __restrict__ sinks, long ldo,
                                                          const float* __restrict__ slopes, int ghead) {
  constexpr int EPT = 4 * VB / NW;               // outputs a thread
  __shared__ __attribute__((aligned(16))) f32x4 Om[NW][16][4 * VB + 1];
  __shared__ float ml[NW][2][16], Ls[16];
  const int tile = gridDim.x - 1 - blockIdx.x;   // later tokens see more keys: start with the long rows
  const int s = tile_seq[tile];
  const int n = qlen[s], tok0 = tile_tok0[tile];
  if (n <= 0 || tok0 >= n) return;               // the whole workgroup (padding tiles)
  const int g = blockIdx.y, R = H / G;
  const int r0 = blockIdx.z * GA_ROWS, Rh = min(GA_ROWS, R - r0);
  const int nq = min(TQ, n - tok0), nrows = nq * Rh;
  const int q0 = qstart[s], p0 = ctx[s] - n;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g4 = lane >> 4;
  const bool row = lr < nrows;                   // rows past nrows are idle: they see no key and are not written
  const long tok = q0 + tok0 + (row ? lr / Rh : 0);
  const int h = g * R + r0 + (row ? lr % Rh : 0);
  const int rpos = row ? p0 + tok0 + lr / Rh : -1, rlo = row ? oldest_key(rpos, win, chunk) : 0;
  const float slp = slopes ? slopes[h] : 0.f;
  f32x4 qf[KB];
  float gv[EPT];
  if (gate)
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int i = threadIdx.x + e * 64 * NW, r = min(i / (16 * VB), nrows - 1), j = min(i % (16 * VB), dv - 1);
      const int hh = g * R + r0 + r % Rh;
      gv[e] = gate[(q0 + tok0 + r / Rh) * ldg + (ghead ? (long)hh : (long)hh * dv + j)];
    }
  const float* qp = q + (tok * H + h) * d;
#pragma unroll
  for (int b = 0; b < KB; ++b) {
    const int i = 16 * b + 4 * g4;
    qf[b] = i < d ? *reinterpret_cast<const f32x4*>(qp + i) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int last = p0 + tok0 + nq - 1, first = oldest_key(p0 + tok0, win, chunk);   // the newest and oldest key any row sees
  const int* btr = bt + (long)s * bt_ld;
  f32x4 kf[KB], vf[VB], kn[KB], vn[VB];
  auto page_of = [&](int k0) { return k0 <= last ? btr[BSZ == 16 ? k0 >> 4 : k0 / BSZ] : 0; };
  auto fetch = [&](int k0, long blk, f32x4 (&k)[KB], f32x4 (&v)[VB]) {   // places past the widths are read at 0: q is 0 there, O is dropped
    const int off = BSZ == 16 ? 0 : k0 % BSZ;
    const float* kp = kc + ((blk * G + g) * BSZ + off + lr) * d;
    const float* vp = vc + (blk * G + g) * dv * BSZ + off + 4 * g4;
#pragma unroll
    for (int b = 0; b < KB; ++b) k[b] = *reinterpret_cast<const f32x4*>(kp + (16 * b + 4 * g4 < d ? 16 * b + 4 * g4 : 0));
#pragma unroll
    for (int b = 0; b < VB; ++b) v[b] = *reinterpret_cast<const f32x4*>(vp + (long)(16 * b + lr < dv ? 16 * b + lr : 0) * BSZ);
  };
  // the wave's next page from k0 on (uniform in the wave): pages between the kept keys and the window are passed over
  auto next = [&](int k0) {
    while (k0 <= last && k0 >= keep && k0 + 16 <= first) k0 += 16 * NW;
    return k0;
  };
  float m = -INFINITY, l = 0.f;
  f32x4 O[VB];
#pragma unroll
  for (int b = 0; b < VB; ++b) O[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  int k0 = next((keep > 0 ? 0 : first / 16 * 16) + 16 * w);
  int k1 = next(k0 + 16 * NW), pg = page_of(k0);
  if (k0 <= last) fetch(k0, pg, kn, vn);
  pg = page_of(k1);            // a page's number is asked for while the one before it is fetched (two rows of 400 keys 17.4 -> 16.2 us)
  while (k0 <= last) {
#pragma unroll
    for (int b = 0; b < KB; ++b) kf[b] = kn[b];
#pragma unroll
    for (int b = 0; b < VB; ++b) vf[b] = vn[b];
    if (k1 <= last) fetch(k1, pg, kn, vn);
    const int k2 = next(k1 + 16 * NW);
    pg = page_of(k2);
    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int x = 0; x < 4; ++x) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][x], qf[b][x], sc, 0, 0, 0);
    bool vis[4];
    float mn = m;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int pk = k0 + 4 * g4 + x;
      vis[x] = pk <= rpos && (pk >= rlo || pk < keep);
      if (cap > 0.f) sc[x] = cap * tanhf(sc[x] / cap);
      else if (slopes) sc[x] -= slp * (float)(rpos - pk);
      if (vis[x]) mn = fmaxf(mn, sc[x]);
    }
    mn = lane_max(mn, 16);
    mn = lane_max(mn, 32);
    const float f = mn > -INFINITY ? expf(m - mn) : 1.f;   // before the first visible key: O and l are 0
    f32x4 p;
    l *= f;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      p[x] = vis[x] ? expf(sc[x] - mn) : 0.f;
      l += p[x];
    }
    m = mn;
    if (k0 + 15 > last) {   // values past the newest key are not of this sequence: whatever they hold, they count as 0
#pragma unroll
      for (int b = 0; b < VB; ++b)
#pragma unroll
        for (int x = 0; x < 4; ++x) vf[b][x] = k0 + 4 * g4 + x <= last ? vf[b][x] : 0.f;
    }
#pragma unroll
    for (int b = 0; b < VB; ++b) {
      O[b] *= f;
#pragma unroll
      for (int x = 0; x < 4; ++x) O[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][x], p[x], O[b], 0, 0, 0);
    }
    k0 = k1;
    k1 = k2;
  }
  l = lane_add(l, 16);
  l = lane_add(l, 32);
  if (g4 == 0) {
    ml[w][0][lr] = m;
    ml[w][1][lr] = l;
  }
  __syncthreads();
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int x = 0; x < NW; ++x) M = fmaxf(M, ml[x][0][lr]);
#pragma unroll
  for (int x = 0; x < NW; ++x) L += ml[x][0][lr] > -INFINITY ? ml[x][1][lr] * expf(ml[x][0][lr] - M) : 0.f;
  const float f = m > -INFINITY ? expf(m - M) : 0.f;
#pragma unroll
  for (int b = 0; b < VB; ++b) Om[w][lr][(16 * b + 4 * g4) / 4] = O[b] * f;
  if (w == 0 && g4 == 0) Ls[lr] = 1.f / (L + (sinks ? expf(sinks[h] - M) : sink > 0.f ? sink * expf(-M) : 0.f));
  __syncthreads();
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int i = threadIdx.x + e * 64 * NW, r = i / (16 * VB), j = i % (16 * VB);
    if (r >= nrows || j >= dv) continue;
    float o = 0.f;
#pragma unroll
    for (int x = 0; x < NW; ++x) o += reinterpret_cast<const float*>(&Om[x][r][0])[j];
    o *= Ls[r];
    if (gate) o *= 1.f / (1.f + expf(-gv[e]));
    out[(q0 + tok0 + r / Rh) * ldo + (long)(g * R + r0 + r % Rh) * dv + j] = o;
  }
}

// ---------------------------------------------------------------- bf16 on the matrix cores
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false)));
  return v;
}
__device__ __forceinline__ float row16_add(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false));
  return v;
}

constexpr int GM_ROWS = 64, GM_KT = 64, GM_BS = 16;   // rows per workgroup, keys per tile, keys per page
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));

// KD >= d, VD >= dv: d is walked in KD / 32 MFMA steps, dv in VD / 16 column blocks; steps and blocks past
// the real widths multiply zeros (a branch around each would drain the matrix pipe).  d % 8 == 0
// (16-byte key rows).
// CAP: the scores are capped at 0 < cap <= CAP_MAX, so exp(score) and its sums stay inside f32 and the
// softmax needs no running maximum (it stays 0) and no rescaling.
// MFMA operand layout (16x16x32): with lr = lane & 15, g4 = lane >> 4, A holds row lr, contraction
// indices 8 g4 .. 8 g4 + 7; B holds column lr, the same indices; the accumulator holds rows
// 4 g4 .. 4 g4 + 3 of column lr.
constexpr float CAP_MAX = 64.f;
// DIST: the scores fall with the distance (`slopes`); the score accumulators start at -slope * distance.
// Up to 64-wide heads four workgroups fit a CU's LDS, and its registers if a wave keeps to 128 (6 sequences of 7300 tokens, 32 / 8 heads:
// 266 us with three, 232 with four).  Up to 192 two must: left alone 192-wide heads took the registers of one (24 decode rows, 8 / 2 heads, 20.0 us
// for 14.2; 3000 tokens under a window of 512 59.6 for 38.8).
template <int KD, int VD, bool CAP, bool DIST>
__global__ void __launch_bounds__(256, KD <= 64 ? 4 : KD <= 192 ? 2 : 1) paged_gqa_mfma_kernel(const u16* __restrict__ q, const u16* __restrict__ kc,
                                                             const u16* __restrict__ vc, const int* __restrict__ bt,
                                                             int bt_ld, const int* __restrict__ qstart,
                                                             const int* __restrict__ qlen, const int* __restrict__ ctx,
                                                             const int* __restrict__ tile_seq,
                                                             const int* __restrict__ tile_tok0, const u16* __restrict__ gate,
                                                             long ldg, u16* __restrict__ out, int H, int G, int d, int dv,
                                                             int TQ, int splits, float* __restrict__ part, int win, int GV,
                                                             float* __restrict__ out32, int keep, float sink, int chunk,
                                                             float cap, const float* __restrict__ sinks, long ldo,
                                                             const float* __restrict__ slopes, int ghead) {
  constexpr int DS = KD / 32, VB = VD / 16, NKB = GM_KT / 16;
  constexpr int KSTR = KD + 8, VSTR = GM_KT + 8, PSTR = GM_KT + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smraw[];
  // key/value heads next to each other: workgroups go round the eight XCDs, so with 8 heads, or a divisor or multiple of it, each XCD
  // walks the keys of its own heads, which its L2 holds (4001 tokens, 16 heads of 96 / 64: 273 -> 187 us; 7300 in six sequences, 8 of 64:
  // 303 -> 255)
  const int g = blockIdx.x % G, tile = (gridDim.x - 1 - blockIdx.x) / G;   // later tokens see more keys: start with the long rows
  const int s = tile_seq[tile];
  const int n = qlen[s];
  const int tok0 = tile_tok0[tile];
  if (n <= 0 || tok0 >= n) return;   // the whole workgroup (padding tiles)
  const int R = H / G;
  const int nq = min(TQ, n - tok0), nrows = nq * R;
  const int q0 = qstart[s], p0 = ctx[s] - n;
  u16* ksh = reinterpret_cast<u16*>(smraw);          // [KT][KSTR]
  u16* vtr = ksh + GM_KT * KSTR;                      // [VD][VSTR]: values transposed, [dim][key]
  u16* pw = vtr + VD * VSTR;                          // [4 waves][hi | lo][16][PSTR]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // in a scalar register: the branches on it are scalar
  const int lr = lane & 15, g4 = lane >> 4;
  u16* phi = pw + wave * (2 * 16 * PSTR);
  u16* plo = phi + 16 * PSTR;
  // row rr -> (token tok0 + rr / R, query head g R + rr % R)
  bf16x8 qa[DS];
  {
    const int row = 16 * wave + lr;
    const bool rk = row < nrows;
    const u16* qp = q + ((long)(q0 + tok0 + (rk ? row / R : 0)) * H + g * R + (rk ? row % R : 0)) * d;
#pragma unroll
    for (int st = 0; st < DS; ++st) {
      const int c = st * 32 + 8 * g4;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (rk && c < d) v = *reinterpret_cast<const uint4*>(qp + c);
      qa[st] = __builtin_bit_cast(bf16x8, v);
    }
  }
  int rpos[4], rlo[4];
  float m[4], l[4], slp[4];
  f32x4 acc[VB];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * wave + 4 * g4 + i;
    rpos[i] = row < nrows ? p0 + tok0 + row / R : -1;     // -1: sees no key
    rlo[i] = row < nrows ? oldest_key(rpos[i], win, chunk) : 0;
    slp[i] = DIST && row < nrows ? slopes[g * R + row % R] : 0.f;
    m[i] = CAP ? 0.f : -INFINITY;
    l[i] = 0.f;
  }
#pragma unroll
  for (int cb = 0; cb < VB; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wave_last = 16 * wave < nrows ? p0 + tok0 + (min(16 * wave + 15, nrows - 1)) / R : -1;
  // the oldest row of the wave; idle rows (past nrows) are masked, so a wave that has any never skips the mask
  const int wave_first = 16 * wave + 15 < nrows ? p0 + tok0 + (16 * wave) / R : -1;
  // the oldest keys the wave's oldest and newest live rows see (a tile wholly before the first is
  // skipped; one not before the second needs no mask at its old end)
  const int wave_lo = 16 * wave < nrows ? oldest_key(p0 + tok0 + (16 * wave) / R, win, chunk) : 0;
  const int wave_lo_last = wave_last >= 0 ? oldest_key(wave_last, win, chunk) : 0;
  // CAP: exponents in base 2
  const float cap2 = cap > 0.f ? (CAP ? 2.88539008f : 2.f) / cap : 0.f;
  const float capl = 1.44269504f * cap;
  const int last = p0 + tok0 + nq - 1;   // the newest key any row sees
  const int* btr = bt + (long)s * bt_ld;
  constexpr int KCH = KD / 8;            // 16-byte chunks of a staged key row
  constexpr int NFK = KD / 32, NFV = VD / 32;      // chunks of K, and of V, a thread moves per tile
  // Score block kb, column lr stands for key 4 lr + kb of the tile (K rows are staged in that order),
  // so a lane's four blocks are four neighbouring keys and its weights leave as 8-byte vectors.
  uint4 pk_[NFK], pv_[NFV];
  // A thread moves the same (key, chunk) and (dim, page, half) of every tile (tiles start at multiples
  // of 64 keys), so only the page ids change from tile to tile: offsets inside a page are kept.
  int koff[NFK], voff[NFV];      // inside a page (past d or dv: the row's first, and zeros when staged)
  int kkey[NFK];
  bool kon[NFK], von[NFV];
  const long kpage = (long)G * GM_BS * d, vpage = (long)GV * dv * GM_BS;
  const int gv = g / (G / GV);
#pragma unroll
  for (int f = 0; f < NFK; ++f) {
    const int e = tid + 256 * f;
    const int kk = e / KCH, c = (e % KCH) * 8;
    kkey[f] = kk;
    kon[f] = c < d;
    koff[f] = (g * GM_BS + (kk & 15)) * d + (kon[f] ? c : 0);
  }
  const int vpg = (tid % (GM_KT / 8)) >> 1;      // the page a thread's values are on
#pragma unroll
  for (int f = 0; f < NFV; ++f) {
    const int e = tid + 256 * f;
    const int j = e / (GM_KT / 8), cc = e % (GM_KT / 8);
    von[f] = j < dv;
    voff[f] = (gv * dv + (von[f] ? j : 0)) * GM_BS + 8 * (cc & 1);
  }
  // A tile's page ids are loaded a tile ahead of its keys, and no load stands behind a condition of its own (pages past the newest key:
  // its page again, and zeros when staged): a load that waits for its page id waits for all loads before it, and a tile took one
  // latency per chunk (us, then -> now: 16 heads of 96 / 64, 4001 tokens 183 -> 143; 16 / 4 of 128, four sequences of 2900 66 -> 54; 16 of 256, 1500
  // tokens 180 -> 121; 32 / 8 of 64, six of 1400 224 -> 211)
  int kid[NFK], vid;
  const int page_last = last >> 4;
  auto fetch_ids = [&](int k0) {
#pragma unroll
    for (int f = 0; f < NFK; ++f) kid[f] = btr[min((k0 + kkey[f]) >> 4, page_last)];
    vid = btr[min((k0 >> 4) + vpg, page_last)];
  };
  auto fetch = [&] {
#pragma unroll
    for (int f = 0; f < NFK; ++f) pk_[f] = *reinterpret_cast<const uint4*>(kc + kid[f] * kpage + koff[f]);
#pragma unroll
    for (int f = 0; f < NFV; ++f) pv_[f] = *reinterpret_cast<const uint4*>(vc + vid * vpage + voff[f]);
  };
  // small grids (decode steps) split a row's key tiles over `splits` workgroups; each leaves its
  // running maximum, sum and unnormalised output in `part`, gqa_combine merges them
  const int tfirst = oldest_key(p0 + tok0, win, chunk) / GM_KT;   // the oldest tile of the window / chunk any row sees
  // kept first keys: their tiles come before the window's in the walk; tile number v of the walk is
  // tile v of the sequence for v < nkeep, else tile tfirst + v - nkeep
  const int nkeep = min(tfirst, (keep + GM_KT - 1) / GM_KT);
  const int ntiles = last / GM_KT + 1 - tfirst + nkeep;
  const int vbeg = (int)((long)ntiles * blockIdx.z / splits);
  const int vend = (int)((long)ntiles * (blockIdx.z + 1) / splits);   // exclusive
  auto tile_k0 = [&](int v) { return (v < nkeep ? v : tfirst + v - nkeep) * GM_KT; };
  if (vbeg < vend) {
    fetch_ids(tile_k0(vbeg));
    fetch();
    fetch_ids(tile_k0(min(vbeg + 1, vend - 1)));
  }
  for (int vt = vbeg; vt < vend; ++vt) {
    const int k0 = tile_k0(vt);
    __syncthreads();   // the previous tile is consumed
    const int nk = last + 1 - k0;
    if (nk < GM_KT || d < KD || dv < VD) {
#pragma unroll
      for (int f = 0; f < NFK; ++f)
        if (!(kon[f] & (kkey[f] < nk))) pk_[f] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int f = 0; f < NFV; ++f)
        if (!(von[f] & (16 * vpg < nk))) pv_[f] = make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int f = 0; f < NFK; ++f) {
      const int e = tid + 256 * f;
      const int kk = e / KCH, c = (e % KCH) * 8;
      *reinterpret_cast<uint4*>(ksh + (16 * (kk & 3) + (kk >> 2)) * KSTR + c) = pk_[f];
    }
#pragma unroll
    for (int f = 0; f < NFV; ++f) {
      const int e = tid + 256 * f;
      const int j = e / (GM_KT / 8), cc = e % (GM_KT / 8);
      *reinterpret_cast<uint4*>(vtr + j * VSTR + 8 * cc) = pv_[f];
    }
    if (vt + 1 < vend) {      // the next tile's loads fly under this tile's products
      fetch();
      fetch_ids(tile_k0(min(vt + 2, vend - 1)));
    }
    __syncthreads();
    if (k0 > wave_last) continue;   // this wave's rows see nothing of the tile (the barriers above are uniform)
    if (k0 >= keep && k0 + GM_KT <= wave_lo) continue;   // ... or the tile lies before every row's window / chunk
    f32x4 sacc[NKB];
    if constexpr (DIST) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float d0 = slp[i] * (float)(k0 + 4 * lr - rpos[i]);
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) sacc[kb][i] = fmaf(slp[i], (float)kb, d0);
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) sacc[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int st = 0; st < DS; ++st) {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        const bf16x8 b = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(ksh + (16 * kb + lr) * KSTR + 8 * g4 + st * 32));
        sacc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[st], b, sacc[kb], 0, 0, 0);
      }
    }
    float sc[NKB][4];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[kb][i] = sacc[kb][i];
    if (!CAP && !DIST && cap > 0.f) {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[kb][i] = cap_fast(sc[kb][i], cap, cap2);
    }
    if constexpr (CAP) {   // log2(e) times the capped score
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sc[kb][i] = capl - 2.f * capl * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(sc[kb][i] * cap2) + 1.f);
    }
    const int key0 = k0 + 4 * lr;
    // a tile inside every row's range needs no mask (wave-uniform, a scalar branch).  The mask is bitwise on
    // purpose, a select per key: written with && and || hipcc made a chain of exec-masked branches of it,
    // and in the 64-wide form dropped the copy of the visible keys' scores
    if (!(k0 + GM_KT - 1 <= wave_first && k0 >= wave_lo_last)) {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + kb;
          const bool vis = (key <= rpos[i]) & ((key >= rlo[i]) | (key < keep));
          sc[kb][i] = vis ? sc[kb][i] : -INFINITY;
        }
    }
    float alpha[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float p[NKB];
      if constexpr (CAP) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          p[kb] = __builtin_amdgcn_exp2f(sc[kb][i]);   // 0 for masked keys
          l[i] += p[kb];
        }
      } else {
        float mx = fmaxf(fmaxf(sc[0][i], sc[1][i]), fmaxf(sc[2][i], sc[3][i]));
        mx = row16_max(mx);
        const float mn = fmaxf(m[i], mx);
        const bool any = mn > -INFINITY;
        alpha[i] = any ? __expf(m[i] - mn) : 1.f;   // m = -inf before the first visible key: 0, and acc, l are 0
        m[i] = mn;
        l[i] *= alpha[i];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          p[kb] = any ? __expf(sc[kb][i] - mn) : 0.f;   // exp(-inf) = 0 for masked keys
          l[i] += p[kb];
        }
      }
      // p = hi + lo with both parts bf16 (the packed conversions round to nearest even)
      const uint32_t h01 = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{p[0], p[1]}, bf16x2v));
      const uint32_t h23 = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{p[2], p[3]}, bf16x2v));
      const f32x2v r01 = {p[0] - __uint_as_float(h01 << 16), p[1] - __uint_as_float(h01 & 0xffff0000u)};
      const f32x2v r23 = {p[2] - __uint_as_float(h23 << 16), p[3] - __uint_as_float(h23 & 0xffff0000u)};
      const uint32_t l01 = __builtin_bit_cast(uint32_t, __builtin_convertvector(r01, bf16x2v));
      const uint32_t l23 = __builtin_bit_cast(uint32_t, __builtin_convertvector(r23, bf16x2v));
      *reinterpret_cast<uint2*>(phi + (4 * g4 + i) * PSTR + 4 * lr) = make_uint2(h01, h23);
      *reinterpret_cast<uint2*>(plo + (4 * g4 + i) * PSTR + 4 * lr) = make_uint2(l01, l23);
    }
    // the patch is this wave's own: its LDS accesses are in order, the fence keeps the compiler's order too
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if constexpr (!CAP) {
      // once the running maxima have settled no row of the wave rescales: skip the sweep over the sums
      if (__any(alpha[0] != 1.f || alpha[1] != 1.f || alpha[2] != 1.f || alpha[3] != 1.f)) {
#pragma unroll
        for (int cb = 0; cb < VB; ++cb)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[cb][i] *= alpha[i];
      }
    }
#pragma unroll
    for (int ks = 0; ks < GM_KT; ks += 32) {
      const bf16x8 ah = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(phi + lr * PSTR + ks + 8 * g4));
      const bf16x8 al = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(plo + lr * PSTR + ks + 8 * g4));
#pragma unroll
      for (int cb = 0; cb < VB; ++cb) {
        const bf16x8 bv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(vtr + (16 * cb + lr) * VSTR + 8 * g4 + ks));
        acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bv, acc[cb], 0, 0, 0);
        acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bv, acc[cb], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float lt = row16_add(l[i]);
    const int row = 16 * wave + 4 * g4 + i;
    if (row >= nrows) continue;
    if (part) {
      float* pr = part + ((((long)tile * G + g) * splits + blockIdx.z) * GM_ROWS + row) * (dv + 2);
      if (lr == 0) { pr[0] = m[i]; pr[1] = lt; }
#pragma unroll
      for (int cb = 0; cb < VB; ++cb)
        if (16 * cb + lr < dv) pr[2 + 16 * cb + lr] = acc[cb][i];
      continue;
    }
    const long tok = q0 + tok0 + row / R;
    const int h = g * R + row % R;
    float inv = 1.f / (lt + (sinks ? __expf(sinks[h] - m[i]) : sink > 0.f ? sink * __expf(-m[i]) : 0.f));
    if (gate && ghead) inv *= 1.f / (1.f + expf(-bf2f(gate[tok * ldg + h])));
#pragma unroll
    for (int cb = 0; cb < VB; ++cb) {
      const int jx = 16 * cb + lr;
      if (jx >= dv) continue;
      float o = acc[cb][i] * inv;
      if (gate && !ghead) o *= 1.f / (1.f + expf(-bf2f(gate[tok * ldg + (long)h * dv + jx])));
      if (out32) out32[tok * ldo + (long)h * dv + jx] = o;
      else out[tok * ldo + (long)h * dv + jx] = f2bf(o);
    }
  }
}

// The same with a row to a lane column:  S^T = K . Q^T  leaves 16 of a tile's scores of one row in a lane, so the row's maximum is eight instructions
// and two lane exchanges where the form above takes seven for each of a lane's four rows, one exponential rescales it, and the weights are at
// once the right operand of  O^T = V^T . P^T  where they went round by LDS.  (Row 16 kb + 4 g + i of the staged keys is key 32 (kb / 2) + 8 g + 4 (kb % 2) + i:
// a lane's scores are then eight neighbouring keys of each half of a tile, as V^T lies.)  Vector instructions bound both forms, two thirds of
// the cycles here: per tile and wave 95 of them and 28 products.  us, above / here: six sequences of 308 to 2600 tokens, 32 / 8 heads of 64 176 / 122,
// with a window of 512 103 / 70; 4001 tokens, 16 heads of 96 / 64 128 / 103; 24 of 160 32.6 / 19.8; four of 200 to 1300, 16 / 4 of 64 with slopes 43 / 29;
// four of 2900, 16 / 4 of 128 429 / 254; 3000, 8 / 2 of 192 / 128 125 / 94.  Two tiles in LDS with one barrier a tile took 139 for 132, chunks
// swizzled for fewer bank conflicts nothing.
template <int KD, int VD, bool CAP, bool DIST>
__global__ void __launch_bounds__(256, KD <= 64 ? 4 : KD <= 96 ? (CAP ? 3 : 4) : 2) gqa_cols_kernel(const u16* __restrict__ q, const u16* __restrict__ kc, const u16* __restrict__ vc,
                                                      const int* __restrict__ bt, int bt_ld, const int* __restrict__ qstart,
                                                      const int* __restrict__ qlen, const int* __restrict__ ctx,
                                                      const int* __restrict__ tile_seq, const int* __restrict__ tile_tok0,
                                                      const u16* __restrict__ gate, long ldg, u16* __restrict__ out, int H, int G, int d,
                                                      int dv, int TQ, int splits, float* __restrict__ part, int win, int keep,
                                                      float sink, int chunk, float cap, const float* __restrict__ sinks, long ldo,
                                                      const float* __restrict__ slopes, int ghead) {
  constexpr int DS = KD / 32, VB = VD / 16, NKB = GM_KT / 16;
  constexpr int KSTR = KD + 8, VSTR = GM_KT + 8;
  constexpr float LOG2E = 1.44269504f;
  __shared__ __attribute__((aligned(16))) u16 ksh[GM_KT * KSTR], vtr[VD * VSTR];      // keys; values transposed, [dim][key]
  const int g = blockIdx.x % G, tile = (gridDim.x - 1 - blockIdx.x) / G;
  const int s = tile_seq[tile];
  const int n = qlen[s];
  const int tok0 = tile_tok0[tile];
  if (n <= 0 || tok0 >= n) return;   // the whole workgroup (padding tiles)
  const int R = H / G;
  const int nq = min(TQ, n - tok0), nrows = nq * R;
  const int q0 = qstart[s], p0 = ctx[s] - n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, g4 = lane >> 4;
  // this lane's row -> (token tok0 + row / R, query head g R + row % R)
  const int row = 16 * wave + lr;
  const bool live = row < nrows;
  const int tl = live ? row / R : 0, h = g * R + (live ? row % R : 0);
  const int rpos = live ? p0 + tok0 + tl : -1, rlo = live ? oldest_key(rpos, win, chunk) : 0;      // -1: sees no key
  const float slp = DIST && live ? slopes[h] : 0.f;
  const long tok = q0 + tok0 + tl;
  bf16x8 qb[DS];
#pragma unroll
  for (int st = 0; st < DS; ++st) {
    const int c = st * 32 + 8 * g4;
    qb[st] = __builtin_bit_cast(bf16x8, live && c < d ? ld16(q + (tok * H + h) * d + c) : make_uint4(0u, 0u, 0u, 0u));
  }
  // The sums hold weights relative to 2^c2, log2 e times the row's maximum m and rounded: what rescales them is how far c2 moves, exactly 1 where the
  // maximum has stayed.  (From m times log2 e unrounded it was off by c2's rounding on every tile: 24000 keys with scores of 100 lost 4e-4 of the oldest keys'
  // weights, here 4e-6, the output's own rounding; time as it was: 153 us for 152 to 155 on the six prompts, 101 for 103 at 96 / 64, 95.6 for
  // 93.2 at 192 / 128.)  Lowest before the first visible key: weights and sums are 0.
  constexpr float LOWEST = -0x1.fffffep127f;
  float m = CAP ? 0.f : -INFINITY, c2 = CAP ? 0.f : LOWEST;
  bool huge = false;      // a maximum that may leave f32's range times log2 e, in any row of the wave: from there on relative to e^m
  // the weights' sum is one more row of  V^T . P^T,  of ones: four products where 16 additions are a twelfth of a tile's vector instructions
  f32x4 l = {0.f, 0.f, 0.f, 0.f};
  // {-1, 0} in a register: as an inline constant the compiler writes it the way the instruction reads {0, -1}
  uint32_t neg = 0xbf80u;
  asm volatile("" : "+s"(neg));
  const bf16x2v minus = __builtin_bit_cast(bf16x2v, neg);
  const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
  f32x4 acc[VB];
#pragma unroll
  for (int cb = 0; cb < VB; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wave_last = 16 * wave < nrows ? p0 + tok0 + (min(16 * wave + 15, nrows - 1)) / R : -1;
  // the oldest row of the wave; idle rows (past nrows) are masked, so a wave that has any never skips the mask
  const int wave_first = 16 * wave + 15 < nrows ? p0 + tok0 + (16 * wave) / R : -1;
  // the oldest keys the wave's oldest and newest live rows see (a tile wholly before the first is
  // skipped; one not before the second needs no mask at its old end)
  const int wave_lo = 16 * wave < nrows ? oldest_key(p0 + tok0 + (16 * wave) / R, win, chunk) : 0;
  const int wave_lo_last = wave_last >= 0 ? oldest_key(wave_last, win, chunk) : 0;
  // CAP: exponents in base 2
  const float cap2 = cap > 0.f ? (CAP ? 2.88539008f : 2.f) / cap : 0.f;
  const float capl = 1.44269504f * cap;
  const int last = p0 + tok0 + nq - 1;   // the newest key any row sees
  const int* btr = bt + (long)s * bt_ld;
  // A wave stages a page of the tile's four: its number is a scalar, and a lane's places in it are the same in every tile.  Page ids are
  // loaded a tile ahead of the keys, and no load stands behind a condition (pages past the newest key: its page again, and zeros when staged).
  constexpr int KCH = KD / 8, NFK = KD / 32, NFV = VD / 32;      // 16-byte chunks of a key row; chunks of K, and of V, a lane moves per tile
  uint4 pk_[NFK], pv_[NFV];
  int koff[NFK], voff[NFV], klds[NFK], kkey[NFK];      // in a page (past d or dv: the row's first, and zeros when staged), in LDS
  bool kon[NFK], von[NFV];
#pragma unroll
  for (int f = 0; f < NFK; ++f) {
    const int e = lane + 64 * f, c = (e % KCH) * 8, kk = 16 * wave + e / KCH;
    kkey[f] = kk;
    kon[f] = c < d;
    koff[f] = (e / KCH) * d + (kon[f] ? c : 0);
    klds[f] = (32 * (kk >> 5) + 16 * ((kk >> 2) & 1) + 4 * ((kk >> 3) & 3) + (kk & 3)) * KSTR + c;
  }
#pragma unroll
  for (int f = 0; f < NFV; ++f) {
    const int j = (lane >> 1) + 32 * f;
    von[f] = j < dv;
    voff[f] = (von[f] ? j : 0) * GM_BS + 8 * (lane & 1);
  }
  const u16 *kg = kc + (long)g * GM_BS * d, *vg = vc + (long)g * dv * GM_BS;
  const long kpage = (long)G * GM_BS * d, vpage = (long)G * dv * GM_BS;
  const int page_last = last >> 4;
  int id;
  auto fetch_ids = [&](int k0) { id = btr[min((k0 >> 4) + wave, page_last)]; };
  auto fetch = [&] {
    const u16 *kp = kg + id * kpage, *vp = vg + id * vpage;
#pragma unroll
    for (int f = 0; f < NFK; ++f) pk_[f] = ld16(kp + koff[f]);
#pragma unroll
    for (int f = 0; f < NFV; ++f) pv_[f] = ld16(vp + voff[f]);
  };
  const int tfirst = oldest_key(p0 + tok0, win, chunk) / GM_KT;   // the oldest tile of the window / chunk any row sees
  const int nkeep = min(tfirst, (keep + GM_KT - 1) / GM_KT);
  const int ntiles = last / GM_KT + 1 - tfirst + nkeep;
  const int vbeg = (int)((long)ntiles * blockIdx.z / splits);
  const int vend = (int)((long)ntiles * (blockIdx.z + 1) / splits);   // exclusive
  auto tile_k0 = [&](int v) { return (v < nkeep ? v : tfirst + v - nkeep) * GM_KT; };
  if (vbeg < vend) {
    fetch_ids(tile_k0(vbeg));
    fetch();
    fetch_ids(tile_k0(min(vbeg + 1, vend - 1)));
  }
  for (int vt = vbeg; vt < vend; ++vt) {
    const int k0 = tile_k0(vt);
    __syncthreads();   // the previous tile is consumed
    const int nk = last + 1 - k0;
    if (nk < GM_KT || d < KD || dv < VD) {
#pragma unroll
      for (int f = 0; f < NFK; ++f)
        if (!(kon[f] & (kkey[f] < nk))) pk_[f] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int f = 0; f < NFV; ++f)
        if (!(von[f] & (16 * wave < nk))) pv_[f] = make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int f = 0; f < NFK; ++f) st16(ksh + klds[f], pk_[f]);
#pragma unroll
    for (int f = 0; f < NFV; ++f) st16(vtr + ((lane >> 1) + 32 * f) * VSTR + 16 * wave + 8 * (lane & 1), pv_[f]);
    if (vt + 1 < vend) {      // the next tile's loads fly under this tile's products
      fetch();
      fetch_ids(tile_k0(min(vt + 2, vend - 1)));
    }
    __syncthreads();
    if (k0 > wave_last) continue;   // this wave's rows see nothing of the tile (the barriers above are uniform)
    if (k0 >= keep && k0 + GM_KT <= wave_lo) continue;   // ... or the tile lies before every row's window / chunk
    const int key0 = k0 + 8 * g4;      // score (kb, i) is of key key0 + 32 (kb / 2) + 4 (kb % 2) + i
    f32x4 sc[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      sc[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (DIST) {
        const float d0 = slp * (float)(key0 + 32 * (kb >> 1) + 4 * (kb & 1) - rpos);
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[kb][i] = fmaf(slp, (float)i, d0);
      }
    }
#pragma unroll
    for (int st = 0; st < DS; ++st)
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, ld16(ksh + (16 * kb + lr) * KSTR + 8 * g4 + st * 32));
        sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qb[st], sc[kb], 0, 0, 0);
      }
    if (!CAP && !DIST && cap > 0.f) {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[kb][i] = cap_fast(sc[kb][i], cap, cap2);
    }
    if constexpr (CAP) {   // log2(e) times the capped score
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sc[kb][i] = capl - 2.f * capl * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(sc[kb][i] * cap2) + 1.f);
    }
    // a tile inside every row's range needs no mask (wave-uniform, a scalar branch; bitwise as above)
    if (!(k0 + GM_KT - 1 <= wave_first && k0 >= wave_lo_last)) {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 32 * (kb >> 1) + 4 * (kb & 1) + i;
          const bool vis = (key <= rpos) & ((key >= rlo) | (key < keep));
          sc[kb][i] = vis ? sc[kb][i] : -INFINITY;
        }
    }
    if constexpr (!CAP) {
      float mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[kb][i]);
      mx = lane_max(mx, 16);
      mx = fmaxf(m, lane_max(mx, 32));
      const float cm = fmaxf(mx * LOG2E, LOWEST);
      if (__any(mx != m)) {      // (once the running maxima have settled no row of the wave rescales; rows that see no key never do)
        huge = huge || __any(fabsf(mx) > 0x1p126f && mx > -INFINITY);
        const float cn = huge ? 0.f : cm;
        const float alpha = mx == m ? 1.f : __builtin_amdgcn_exp2f(huge ? (m - mx) * LOG2E : c2 - cn);
        m = mx;
        c2 = cn;
        l *= alpha;
#pragma unroll
        for (int cb = 0; cb < VB; ++cb) acc[cb] *= alpha;
      }
      if (__builtin_expect(huge, 0)) {
        const float mf = fmaxf(m, LOWEST);
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[kb][i] -= mf;
      }
    }
    bf16x8 ph[NKB / 2], pl[NKB / 2];      // p = hi + lo with both parts bf16 (the packed conversions round to nearest even)
#pragma unroll
    for (int ks = 0; ks < NKB / 2; ++ks) {
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = sc[2 * ks + (j >> 2)][j & 3];
        p[j] = __builtin_amdgcn_exp2f(CAP ? x : fmaf(x, LOG2E, -c2));      // exp(-inf) = 0 for masked keys
      }
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hi[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{p[2 * j], p[2 * j + 1]}, bf16x2v));
        const bf16x2v hb = __builtin_bit_cast(bf16x2v, hi[j]);
        const f32x2v r = {__builtin_amdgcn_fdot2_f32_bf16(hb, minus, p[2 * j], false),
                          __builtin_amdgcn_fdot2_f32_bf16(hb, bf16x2v{0.f, -1.f}, p[2 * j + 1], false)};      // p - hi, exact
        lo[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2v));
      }
      ph[ks] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
      pl[ks] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
    }
    __builtin_amdgcn_s_setprio(1);      // (ahead of the other waves' vector instructions: 132 -> 122 us)
#pragma unroll
    for (int ks = 0; ks < NKB / 2; ++ks) {
      if constexpr (VB <= 4) {
        bf16x8 v[VB];
#pragma unroll
        for (int cb = 0; cb < VB; ++cb) v[cb] = __builtin_bit_cast(bf16x8, ld16(vtr + (16 * cb + lr) * VSTR + 8 * g4 + 32 * ks));
        l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, ph[ks], l, 0, 0, 0);
#pragma unroll
        for (int cb = 0; cb < VB; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[cb], ph[ks], acc[cb], 0, 0, 0);
        l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pl[ks], l, 0, 0, 0);
#pragma unroll
        for (int cb = 0; cb < VB; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[cb], pl[ks], acc[cb], 0, 0, 0);
      } else {      // (with all of eight blocks' values at hand 304 us for 255)
        l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, ph[ks], l, 0, 0, 0);
        l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pl[ks], l, 0, 0, 0);
#pragma unroll
        for (int cb = 0; cb < VB; ++cb) {
          const bf16x8 v = __builtin_bit_cast(bf16x8, ld16(vtr + (16 * cb + lr) * VSTR + 8 * g4 + 32 * ks));
          acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, ph[ks], acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pl[ks], acc[cb], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  if (!live) return;
  if (part) {      // relative to e^m, as what merges them takes them
    float* pr = part + ((((long)tile * G + g) * splits + blockIdx.z) * GM_ROWS + row) * (dv + 2);
    const float f = CAP || huge || !(m > -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(-fmaf(m, LOG2E, -c2));
    if (g4 == 0) { pr[0] = m; pr[1] = l[0] * f; }
#pragma unroll
    for (int cb = 0; cb < VB; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * cb + 4 * g4 + i < dv) pr[2 + 16 * cb + 4 * g4 + i] = acc[cb][i] * f;
    return;
  }
  auto weight = [&](float x) { return huge ? __expf(x - m) : __builtin_amdgcn_exp2f(fmaf(x, LOG2E, -c2)); };
  float inv = 1.f / (l[0] + (sinks ? weight(sinks[h]) : sink > 0.f ? sink * weight(0.f) : 0.f));
  if (gate && ghead) inv *= 1.f / (1.f + expf(-bf2f(gate[tok * ldg + h])));
  auto recip = [](float x) { const float r = __builtin_amdgcn_rcpf(x); return x < 1e38f ? r * fmaf(-x, r, 2.f) : r; };
  const u16* gr = gate && !ghead ? gate + tok * ldg + (long)h * dv : nullptr;
  u16* o = out + tok * ldo + (long)h * dv;
  const bool whole = dv % 4 == 0 && ldo % 4 == 0 && ldg % 4 == 0 && (((uintptr_t)out | (uintptr_t)gate) & 7) == 0;      // four outputs at a time
#pragma unroll
  for (int cb = 0; cb < VB; ++cb) {
    const int j = 16 * cb + 4 * g4;
    u16x4 y;
    if (whole && j < dv) {
      const u16x4 z = gr ? *reinterpret_cast<const u16x4*>(gr + j) : u16x4{};
#pragma unroll
      for (int i = 0; i < 4; ++i) y.v[i] = f2bf(acc[cb][i] * inv * (gr ? recip(1.f + expf(-bf2f(z.v[i]))) : 1.f));
      *reinterpret_cast<u16x4*>(o + j) = y;
    } else
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j + i < dv) o[j + i] = f2bf(acc[cb][i] * inv * (gr ? recip(1.f + expf(-bf2f(gr[j + i]))) : 1.f));
  }
}

// The same for few rows a tile (decode steps: a token's R <= 16 heads): there paged_gqa_mfma has one wave of four with live rows, which
// walks every tile of its split behind two barriers (3 us a tile).  Here each wave takes 32-key chunks of its own and keeps its own
// maximum, sum and O^T; keys and values come from the pages straight to registers, the next chunk's while this one is multiplied, and
// no barrier stands before the waves meet at the end.  S^T = K . Q^T leaves a head's scores in one lane column, P^T feeds
// O^T = V^T . P^T with the key order 8 g + j <-> j < 4 ? 4 g + j : 16 + 4 g + j - 4 (two 8-byte loads of V^T's pages); p = hi + lo as
// above.  With splits 16, merge included: four sequences of 1300, 8 heads of 64 with slopes 19 -> 13 us; six of 2600, 8 splits 28 -> 19.
// More than 16 rows (a tile of a short portion) are walked 16 at a time.
template <int KD, int VD, bool CAP, bool DIST>
__global__ void __launch_bounds__(256, 2) gqa_few_kernel(const u16* __restrict__ q, const u16* __restrict__ kc, const u16* __restrict__ vc,
                                                      const int* __restrict__ bt, int bt_ld, const int* __restrict__ qstart,
                                                      const int* __restrict__ qlen, const int* __restrict__ ctx,
                                                      const int* __restrict__ tile_seq, const int* __restrict__ tile_tok0,
                                                      const u16* __restrict__ gate, long ldg, u16* __restrict__ out, int H, int G, int d,
                                                      int dv, int TQ, int splits, float* __restrict__ part, int win, int keep,
                                                      float sink, int chunk, float cap, const float* __restrict__ sinks, long ldo,
                                                      const float* __restrict__ slopes, int ghead) {
  constexpr int KU = KD / 32, VB = VD / 16;
  __shared__ __attribute__((aligned(16))) f32x4 Om[4][VB * 64];
  __shared__ float ml[4][2][16];
  const int g = blockIdx.x % G, tile = blockIdx.x / G;
  const int s = tile_seq[tile], tok0 = tile_tok0[tile];
  const int n = qlen[s], q0 = qstart[s], p0 = ctx[s] - n;
  if (n <= 0 || tok0 >= n) return;   // the whole workgroup (padding tiles)
  const int R = H / G, nq = min(TQ, n - tok0), nrows = nq * R;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, g4 = lane >> 4;
  const int last = p0 + tok0 + nq - 1;   // the newest key any row sees
  const int* btr = bt + (long)s * bt_ld;
  const float cap2 = cap > 0.f ? (CAP ? 2.88539008f : 2.f) / cap : 0.f, capl = 1.44269504f * cap;
  // the walk over tiles of 64 keys and its splits: as in paged_gqa_mfma
  const int tfirst = oldest_key(p0 + tok0, win, chunk) / GM_KT, nkeep = min(tfirst, (keep + GM_KT - 1) / GM_KT);
  const int ntiles = last / GM_KT + 1 - tfirst + nkeep;
  const int vbeg = (int)((long)ntiles * blockIdx.z / splits), nch = 2 * ((int)((long)ntiles * (blockIdx.z + 1) / splits) - vbeg);
  auto key0 = [&](int c) { const int v = vbeg + (c >> 1); return (v < nkeep ? v : tfirst + v - nkeep) * GM_KT + 32 * (c & 1); };
  struct Pages { int a, b; };
  auto pages = [&](int c) {
    Pages pg{0, 0};
    if (c < nch) {
      const int k0 = key0(c);
      if (k0 <= last) pg.a = btr[k0 >> 4];
      if (k0 + 16 <= last) pg.b = btr[(k0 >> 4) + 1];
    }
    return pg;
  };
  const u16* kl = kc + ((long)g * GM_BS + lr) * d + 8 * g4;
  const u16* vl = vc + ((long)g * dv + lr) * GM_BS + 4 * g4;
  const long kpage = (long)G * GM_BS * d, vpage = (long)G * dv * GM_BS;
  struct Keys { uint4 k[2][KU]; uint2 v[2][VB]; };
  auto load = [&](Keys& x, int c, Pages pg) {      // pages past the last key read as zeros
    const int k0 = key0(c);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bool on = k0 + 16 * t <= last;
      const long page = t ? pg.b : pg.a;
#pragma unroll
      for (int u = 0; u < KU; ++u) x.k[t][u] = on && 32 * u + 8 * g4 < d ? ld16(kl + page * kpage + 32 * u) : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int b = 0; b < VB; ++b)
        x.v[t][b] = on && 16 * b + lr < dv ? *reinterpret_cast<const uint2*>(vl + page * vpage + 16 * b * GM_BS) : make_uint2(0u, 0u);
    }
  };
  for (int rb = 0; rb < nrows; rb += 16) {
    const int row = rb + lr;
    const bool live = row < nrows;
    const int tl = live ? row / R : 0, h = g * R + (live ? row % R : 0);
    const int rpos = live ? p0 + tok0 + tl : -1, rlo = live ? oldest_key(rpos, win, chunk) : 0;
    const float slp = DIST && live ? slopes[h] : 0.f;
    const long tok = q0 + tok0 + tl;
    Pages pg = pages(wave);
    bf16x8 qf[KU];
#pragma unroll
    for (int u = 0; u < KU; ++u)
      qf[u] = __builtin_bit_cast(bf16x8, live && 32 * u + 8 * g4 < d ? ld16(q + (tok * H + h) * d + 32 * u + 8 * g4) : make_uint4(0u, 0u, 0u, 0u));
    float m = CAP ? 0.f : -INFINITY, l = 0.f;
    f32x4 O[VB];
#pragma unroll
    for (int b = 0; b < VB; ++b) O[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    Keys cur, nxt;
    if (wave < nch) load(cur, wave, pg);
    pg = pages(wave + 4);
    for (int c = wave; c < nch; c += 4) {
      if (c + 4 < nch) load(nxt, c + 4, pg);
      pg = pages(c + 8);
      const int k0 = key0(c);
      float p[8];
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 sc = {0.f, 0.f, 0.f, 0.f};
        if constexpr (DIST)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[i] = slp * (float)(k0 + 16 * t + 4 * g4 + i - rpos);
#pragma unroll
        for (int u = 0; u < KU; ++u) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, cur.k[t][u]), qf[u], sc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = sc[i];
          if (!CAP && !DIST && cap > 0.f) v = cap_fast(v, cap, cap2);
          if constexpr (CAP) v = capl - 2.f * capl * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v * cap2) + 1.f);
          const int key = k0 + 16 * t + 4 * g4 + i;
          const bool vis = (key <= rpos) & ((key >= rlo) | (key < keep));
          v = vis ? v : -INFINITY;
          p[4 * t + i] = v;
          mx = fmaxf(mx, v);
        }
      }
      float alpha = 1.f;
      if constexpr (CAP) {
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = __builtin_amdgcn_exp2f(p[j]);   // 0 for masked keys
      } else {
        mx = lane_max(mx, 16);
        mx = lane_max(mx, 32);
        const float mn = fmaxf(m, mx);
        const bool any = mn > -INFINITY;
        alpha = any ? __expf(m - mn) : 1.f;   // m = -inf before the first visible key: 0, and O, l are 0
        m = mn;
        l *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = any ? __expf(p[j] - mn) : 0.f;
#pragma unroll
        for (int b = 0; b < VB; ++b) O[b] *= alpha;
      }
      float lo[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        l += p[j];
        lo[j] = p[j] - bf2f(f2bf(p[j]));
      }
      const bf16x8 ph = __builtin_bit_cast(bf16x8, pack8(p)), pl = __builtin_bit_cast(bf16x8, pack8(lo));
      if (k0 + 31 > last) {      // values behind the last key: whatever an earlier sequence left, and 0 times an infinity is NaN
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int left = last + 1 - (k0 + 16 * t + 4 * g4);      // of this lane's four keys
          const unsigned x = left >= 2 ? ~0u : left == 1 ? 0xffffu : 0u, y = left >= 4 ? ~0u : left == 3 ? 0xffffu : 0u;
#pragma unroll
          for (int b = 0; b < VB; ++b) { cur.v[t][b].x &= x; cur.v[t][b].y &= y; }
        }
      }
#pragma unroll
      for (int b = 0; b < VB; ++b) {
        const bf16x8 vf = __builtin_bit_cast(bf16x8, make_uint4(cur.v[0][b].x, cur.v[0][b].y, cur.v[1][b].x, cur.v[1][b].y));
        O[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph, O[b], 0, 0, 0);
        O[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, O[b], 0, 0, 0);
      }
      cur = nxt;
    }
    l = lane_add(l, 16);
    l = lane_add(l, 32);
    if (g4 == 0) { ml[wave][0][lr] = m; ml[wave][1][lr] = l; }
#pragma unroll
    for (int b = 0; b < VB; ++b) Om[wave][b * 64 + lane] = O[b];
    __syncthreads();
    float M = ml[0][0][lr], L = 0.f, f[4];
#pragma unroll
    for (int x = 1; x < 4; ++x) M = fmaxf(M, ml[x][0][lr]);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      f[x] = CAP ? 1.f : ml[x][0][lr] > -INFINITY ? __expf(ml[x][0][lr] - M) : 0.f;
      L += ml[x][1][lr] * f[x];
    }
    if (live) {
      float* pr = part ? part + ((((long)tile * G + g) * splits + blockIdx.z) * GM_ROWS + row) * (dv + 2) : nullptr;
      if (pr && wave == 0 && g4 == 0) { pr[0] = M; pr[1] = L; }
      float inv = 1.f;
      if (!pr) {
        inv = 1.f / (L + (sinks ? __expf(sinks[h] - M) : sink > 0.f ? sink * __expf(-M) : 0.f));
        if (gate && ghead) inv *= 1.f / (1.f + expf(-bf2f(gate[tok * ldg + h])));
      }
#pragma unroll
      for (int y = 0; y < (VB + 3) / 4; ++y) {
        const int b = wave + 4 * y;
        if (b >= VB) break;
        const f32x4 o = (Om[0][b * 64 + lane] * f[0] + Om[1][b * 64 + lane] * f[1]) + (Om[2][b * 64 + lane] * f[2] + Om[3][b * 64 + lane] * f[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = 16 * b + 4 * g4 + i;
          if (j >= dv) continue;
          if (pr) {
            pr[2 + j] = o[i];
            continue;
          }
          float v = o[i] * inv;
          if (gate && !ghead) v *= 1.f / (1.f + expf(-bf2f(gate[tok * ldg + (long)h * dv + j])));
          out[tok * ldo + (long)h * dv + j] = f2bf(v);
        }
      }
    }
    __syncthreads();
  }
}

// merge the key splits of paged_gqa_mfma: one wave per (tile, kv head, row)
__global__ void __launch_bounds__(256) gqa_combine_kernel(const float* __restrict__ part, int splits,
                                                          const int* __restrict__ qstart, const int* __restrict__ qlen,
                                                          const int* __restrict__ tile_seq,
                                                          const int* __restrict__ tile_tok0, const u16* __restrict__ gate,
                                                          long ldg, u16* __restrict__ out, int H, int G, int dv, int TQ,
                                                          float* __restrict__ out32, float sink,
                                                          const float* __restrict__ sinks, long ldo, int ghead) {
  // the first row's partials are asked for before it is known that there is such a row (every row has its place), and with their
  // weights: this is bound by trips to memory one behind the other (four users, 16 splits: 6.0 -> 4.6 us)
  constexpr int NZ = 16;
  const int g = blockIdx.y, R = H / G, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long zs = (long)GM_ROWS * (dv + 2);
  const float* pt = part + ((long)blockIdx.x * G + g) * splits * zs;
  int row = blockIdx.z * 4 + wave;
  float mz = -INFINITY, lz = 0.f, first[NZ];
  auto stats = [&] {      // lane z holds split z's maximum and sum (splits <= 64); weights travel by shuffles
    const float* pr = pt + (long)row * (dv + 2);
    mz = lane < splits ? pr[lane * zs] : -INFINITY;
    lz = lane < splits ? pr[lane * zs + 1] : 0.f;
  };
  if (row < GM_ROWS) {
    stats();
#pragma unroll
    for (int z = 0; z < NZ; ++z) first[z] = z < splits && lane < dv ? pt[z * zs + (long)row * (dv + 2) + 2 + lane] : 0.f;
  }
  const int s = tile_seq[blockIdx.x];
  const int n = qlen[s], tok0 = tile_tok0[blockIdx.x], q0 = qstart[s];
  if (n <= 0 || tok0 >= n) return;
  const int nrows = min(TQ, n - tok0) * R;
  for (bool ahead = true; row < nrows; row += 4 * gridDim.z, ahead = false) {
    const float* pr = pt + (long)row * (dv + 2);
    if (!ahead) stats();
    const float M = wave_max(mz);
    const float wz = mz > -INFINITY ? expf(mz - M) : 0.f;
    const long tok = q0 + tok0 + row / R;
    const int h = g * R + row % R;
    const float L = wave_sum(lz * wz) + (sinks ? expf(sinks[h] - M) : sink > 0.f ? sink * expf(-M) : 0.f);
    for (int j0 = 0; j0 < dv; j0 += 64) {     // every lane stays in the loop: the shuffles read all lanes
      const int jx = j0 + lane;
      const bool on = jx < dv;
      float o = 0.f;
      int z0 = 0;
      if (ahead && j0 == 0) {
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
          const float w = __shfl(wz, z, 64);
          if (z < splits) o += first[z] * w;
        }
        z0 = min(splits, NZ);
      }
#pragma unroll 4
      for (int z = z0; z < splits; ++z) {
        const float w = __shfl(wz, z, 64);
        if (on) o += pr[z * zs + 2 + jx] * w;
      }
      if (!on) continue;
      o /= L;
      if (gate) o *= 1.f / (1.f + expf(-bf2f(gate[tok * ldg + (ghead ? (long)h : (long)h * dv + jx)])));
      if (out32) out32[tok * ldo + (long)h * dv + jx] = o;
      else out[tok * ldo + (long)h * dv + jx] = f2bf(o);
    }
  }
}

long gqa_mfma_lds(int KD, int VD) { return 2L * (GM_KT * (KD + 8) + (long)VD * (GM_KT + 8) + 4L * 2 * 16 * (GM_KT + 8)); }

long gqa_lds(int d, int dv, int KT) { return 4L * (GA_ROWS * d + (long)KT * (d | 1) + (long)KT * dv + GA_ROWS * 64); }

#define ENSURE_LDS(kernel, bytes)                                                                          \
  do {                                                                                                     \
    static long have_ = 48 * 1024;                                                                         \
    if ((bytes) > have_) {                                                                                 \
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(bytes)); \
      have_ = (bytes);                                                                                     \
    }                                                                                                      \
  } while (0)

template <typename T, int NJ>
int launch_gqa(dim3 grid, long lds, hipStream_t st, const T* q, const T* kc, const T* vc, const int* bt, int bt_ld, int BSZ,
               const int* qstart, const int* qlen, const int* ctx, const int* tile_seq, const int* tile_tok0, const T* gate,
               long ldg, T* out, int H, int G, int d, int dv, int TQ, int KT, int win, int GV, float* out32, int keep,
               float sink, int chunk, float cap, const float* sinks, long ldo, const float* slopes, int ghead) {
  ENSURE_LDS((paged_gqa_kernel<T, NJ>), lds);
  hipLaunchKernelGGL((paged_gqa_kernel<T, NJ>), grid, dim3(256), lds, st, q, kc, vc, bt, bt_ld, BSZ, qstart, qlen, ctx, tile_seq,
                     tile_tok0, gate, ldg, out, H, G, d, dv, TQ, KT, win, GV, out32, keep, sink, chunk, cap, sinks, ldo, slopes,
                     ghead);
  return (int)hipGetLastError();
}

template <typename T>
int launch_gqa_t(int nj, dim3 grid, long lds, hipStream_t st, const void* q, const void* kc, const void* vc, const int* bt,
                 int bt_ld, int BSZ, const int* qstart, const int* qlen, const int* ctx, const int* tile_seq,
                 const int* tile_tok0, const void* gate, long ldg, void* out, int H, int G, int d, int dv, int TQ, int KT,
                 int win, int GV, float* out32, int keep, float sink, int chunk, float cap, const float* sinks, long ldo,
                 const float* slopes, int ghead) {
#define GQA(NJ) return launch_gqa<T, NJ>(grid, lds, st, (const T*)q, (const T*)kc, (const T*)vc, bt, bt_ld, BSZ, qstart, qlen, ctx, tile_seq, tile_tok0, (const T*)gate, ldg, (T*)out, H, G, d, dv, TQ, KT, win, GV, out32, keep, sink, chunk, cap, sinks, ldo, slopes, ghead)
  if (nj <= 1) GQA(1);
  if (nj <= 2) GQA(2);
  GQA(4);
#undef GQA
}

}  // namespace

extern "C" int dllm_attn_prep(const void* proj, long ld, int f32, int H, int G, int d, int dv, const float* cos_sin,
                              int tab_w, int rot, float eps, const float* qscale, const int* pos, const int* slots, void* kc,
                              void* vc, void* q, long T, int BSZ, void* zero_rows, int zw, hipStream_t st) {
  if (T <= 0) return 0;
  if (rot < 0 || rot > d || (rot & 1) || rot > tab_w) return -1;
  uint32_t* const z = (uint32_t*)zero_rows;
  // whole vectors: heads of 32 to 256, halves of the rotation and values in eights, 16-byte aligned rows; and enough of them: 16 tokens a
  // workgroup leave few steps' worth of waves, of which each waits for all its loads (element by element / here, us, heads + key heads
  // x width: 40 x 64, 6 tokens 3.2 / 4.0, 64 3.8 / 5.8, 192 5.4 / 5.9, 256 6.3 / 6.0; 20 x 64, 384 5.4 / 5.9, 512 6.4 / 6.0; 5 x 256, 700 6.0 / 6.3,
  // 1500 9.3 / 7.9; 32 x 128, 128 4.5 / 5.0, 192 5.4 / 5.2)
  if (T * (H + G) * (d + 128) >= 2000000 && !f32 && (d == 32 || d == 64 || d == 128 || d == 256) && dv % 8 == 0 && rot % 16 == 0 && ld % 8 == 0 && tab_w % 4 == 0 && T < (1 << 20) &&
      (((uintptr_t)proj | (uintptr_t)cos_sin | (uintptr_t)kc | (uintptr_t)q) & 15) == 0) {
    const int ny = ((H + G) * (d / 8) + 63) / 64;
    const dim3 g(((unsigned)T + APV_T - 1) / APV_T, ny + (G * dv + APV_V - 1) / APV_V);
#define APV(D)                                                                                                                     \
  hipLaunchKernelGGL(attn_prep_vec_kernel<D>, g, dim3(256), 0, st, (const u16*)proj, ld, H, G, dv, cos_sin, tab_w, rot, eps, qscale, pos, \
                     slots, (u16*)kc, (u16*)vc, (u16*)q, BSZ, (int)T, ny, z, zw)
    if (d == 32) APV(32);
    else if (d == 64) APV(64);
    else if (d == 128) APV(128);
    else APV(256);
#undef APV
    return (int)hipGetLastError();
  }
  const dim3 grid((unsigned)T, (H + G + 3) / 4);
  if (f32)
    hipLaunchKernelGGL(attn_prep_kernel<float>, grid, dim3(256), 0, st, (const float*)proj, ld, H, G, d, dv, cos_sin, tab_w, rot,
                       eps, qscale, pos, slots, (float*)kc, (float*)vc, (float*)q, BSZ, z, zw);
  else
    hipLaunchKernelGGL(attn_prep_kernel<u16>, grid, dim3(256), 0, st, (const u16*)proj, ld, H, G, d, dv, cos_sin, tab_w, rot, eps,
                       qscale, pos, slots, (u16*)kc, (u16*)vc, (u16*)q, BSZ, z, zw);
  return (int)hipGetLastError();
}

// The matrix-core form takes bf16, 16-key pages, key rows of whole 16-byte vectors, widths <= 256 and
// at most 64 query heads per key/value head.
extern "C" int dllm_gqa_mfma_ok(int f32, int H, int G, int d, int dv, int BSZ) {
  return !f32 && BSZ == GM_BS && G >= 1 && H % G == 0 && H / G <= GM_ROWS && d % 8 == 0 && d <= 256 && dv <= 256 && d >= 8;
}

// tokens one workgroup covers for H / G query heads per key/value head
extern "C" int dllm_gqa_tile_tokens(int H, int G, int mfma) {
  const int R = H / G, rows = mfma ? GM_ROWS : GA_ROWS;
  return R >= rows ? 1 : rows / R;
}

extern "C" int dllm_paged_gqa(const void* q, const void* kc, const void* vc, int f32, const int* bt, int bt_ld, int BSZ,
                              const int* qstart, const int* qlen, const int* ctx, const int* tile_seq, const int* tile_tok0,
                              int n_tiles, const void* gate, long ldg, void* out, int H, int G, int d, int dv, int mfma,
                              int splits, float* part, int win, int GV, int out_f32, int keep, float sink, int chunk, float cap,
                              const float* sinks, long ldo, const float* slopes, int ghead, long T, hipStream_t st) {
  if (n_tiles <= 0) return 0;
  if (slopes && cap > 0.f) return -1;
  if (chunk < 0 || (chunk > 0 && win > 0) || cap < 0.f || ldo < (long)H * dv) return -1;
  if (G < 1 || H % G || dv > 256 || d < 1 || GV < 1 || G % GV || win < 0 || keep < 0 || sink < 0.f) return -1;
  if (win <= 0 && chunk <= 0) keep = 0;     // without a bound every key is seen anyway
  float* out32 = out_f32 ? (float*)out : nullptr;
  if (mfma) {
    if (!dllm_gqa_mfma_ok(f32, H, G, d, dv, BSZ)) return -1;
    if (splits < 1 || (splits > 1 && !part)) return -1;
    const dim3 grid((unsigned)n_tiles * G, 1, splits);
    const int TQ = dllm_gqa_tile_tokens(H, G, 1);
    float* pp = splits > 1 ? part : nullptr;
#define GQT(KD, VD, CAP, DIST)                                                                                           \
  do {                                                                                                                   \
    const long lds = gqa_mfma_lds(KD, VD);                                                                               \
    ENSURE_LDS((paged_gqa_mfma_kernel<KD, VD, CAP, DIST>), lds);                                                         \
    hipLaunchKernelGGL((paged_gqa_mfma_kernel<KD, VD, CAP, DIST>), grid, dim3(256), lds, st, (const u16*)q, (const u16*)kc, \
                       (const u16*)vc, bt, bt_ld, qstart, qlen, ctx, tile_seq, tile_tok0, (const u16*)gate, ldg,         \
                       (u16*)out, H, G, d, dv, TQ, splits, pp, win, GV, out32, keep, sink, chunk, cap, sinks, ldo,       \
                       slopes, ghead);                                                                                   \
  } while (0)
    // keys wider than the values (latent attention on expanded keys: unrotated and rotated parts) have forms
    // of their own, so that the extra dims do not widen the value side
#define GQZ(CAP, DIST)                                                                                                   \
  do {                                                                                                                   \
    if (d <= 64 && dv <= 64) GQT(64, 64, CAP, DIST);                                                                     \
    else if (d <= 96 && dv <= 64) GQT(96, 64, CAP, DIST);                                                                \
    else if (d <= 128 && dv <= 128) GQT(128, 128, CAP, DIST);                                                            \
    else if (d <= 192 && dv <= 128) GQT(192, 128, CAP, DIST);                                                            \
    else GQT(256, 256, CAP, DIST);                                                                                       \
  } while (0)
    // at most 16 rows a tile on average: decode steps.  (Heads of a group of one with fewer than 100 keys take up to 1.6 us longer than as tiles,
    // 64 sequences of 64 8.0 / 9.6; 200 keys 16.6 / 12.7.)  Not where key heads share their values or the result is f32: those are the maps
    // of differential attention, whose difference keeps the order of sums of paged_gqa_mfma
    if (GV == G && !out32 && d <= 128 && dv <= 128 && T * (H / G) <= 16L * n_tiles) {
#define GQM(KD, VD, CAP, DIST)                                                                                                   \
  hipLaunchKernelGGL((gqa_few_kernel<KD, VD, CAP, DIST>), grid, dim3(256), 0, st, (const u16*)q, (const u16*)kc, (const u16*)vc, bt, \
                     bt_ld, qstart, qlen, ctx, tile_seq, tile_tok0, (const u16*)gate, ldg, (u16*)out, H, G, d, dv, TQ, splits, pp, win, keep, \
                     sink, chunk, cap, sinks, ldo, slopes, ghead)
#define GQF(CAP, DIST)                                 \
  do {                                                 \
    if (d <= 64 && dv <= 64) GQM(64, 64, CAP, DIST);   \
    else GQM(128, 128, CAP, DIST);                     \
  } while (0)
      if (cap > 0.f && cap <= CAP_MAX) GQF(true, false);
      else if (slopes) GQF(false, true);
      else GQF(false, false);
#undef GQF
#undef GQM
    } else if (GV == G && !out32 && d <= 192 && dv <= 128) {      // (wider heads' accumulators and keys take more registers than a wave has)
#define GQC(KD, VD, CAP, DIST)                                                                                                    \
  hipLaunchKernelGGL((gqa_cols_kernel<KD, VD, CAP, DIST>), grid, dim3(256), 0, st, (const u16*)q, (const u16*)kc, (const u16*)vc, bt, \
                     bt_ld, qstart, qlen, ctx, tile_seq, tile_tok0, (const u16*)gate, ldg, (u16*)out, H, G, d, dv, TQ, splits, pp, win, keep, \
                     sink, chunk, cap, sinks, ldo, slopes, ghead)
#define GQL(CAP, DIST)                                         \
  do {                                                         \
    if (d <= 64 && dv <= 64) GQC(64, 64, CAP, DIST);           \
    else if (d <= 96 && dv <= 64) GQC(96, 64, CAP, DIST);      \
    else if (d <= 128 && dv <= 128) GQC(128, 128, CAP, DIST);  \
    else GQC(192, 128, CAP, DIST);                             \
  } while (0)
      if (cap > 0.f && cap <= CAP_MAX) GQL(true, false);
      else if (slopes) GQL(false, true);
      else GQL(false, false);
#undef GQL
#undef GQC
    } else if (cap > 0.f && cap <= CAP_MAX) GQZ(true, false);
    else if (slopes) GQZ(false, true);
    else GQZ(false, false);
#undef GQZ
#undef GQT
    if (pp) {
      // a wave asks for its row's partials before it knows that there is such a row, so the launch has waves for four times the rows that
      // tiles have on average (all of a decode step's) and goes round where a tile has more.  With waves for every row a tile could
      // have, their loads cost more than they hide: 64 sequences of 100 keys, 16 heads of 64 on 4, two splits 14.9 us, here 11.8
      const int R = H / G, full = TQ * R < GM_ROWS ? TQ * R : GM_ROWS;
      const long rows = T <= n_tiles ? R : 4 * ((T * R + n_tiles - 1) / n_tiles);
      hipLaunchKernelGGL(gqa_combine_kernel, dim3(n_tiles, G, (unsigned)((rows < full ? rows : full) + 3) / 4), dim3(256), 0, st, pp, splits, qstart, qlen,
                         tile_seq, tile_tok0, (const u16*)gate, ldg, (u16*)out, H, G, dv, TQ, out32, sink, sinks, ldo, ghead);
    }
    return (int)hipGetLastError();
  }
  // f32, whole pages of 16 keys, key and query rows of whole 16-byte vectors: the matrix cores.  Not where key heads share their
  // values: those are the maps of differential attention, whose difference keeps the order of sums of paged_gqa
  if (f32 && GV == G && BSZ % 16 == 0 && d % 4 == 0 && d <= 128 && dv <= 128 && (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) & 15) == 0) {
    const dim3 g3(n_tiles, G, (H / G + GA_ROWS - 1) / GA_ROWS);
    const int tq = dllm_gqa_tile_tokens(H, G, 0);
    const bool wide = (long)g3.x * g3.y * g3.z <= GQF_WIDE;
#define GQF2(KB, VB, NW)                                                                                                     \
  hipLaunchKernelGGL((gqa_f32_kernel<KB, VB, NW>), g3, dim3(64 * NW), 0, st, (const float*)q, (const float*)kc, (const float*)vc, bt, \
                     bt_ld, BSZ, qstart, qlen, ctx, tile_seq, tile_tok0, (const float*)gate, ldg, (float*)out, H, G, d, dv, tq, win,  \
                     keep, sink, chunk, cap, sinks, ldo, slopes, ghead)
#define GQF(KB, VB)                        \
  do {                                     \
    if (wide) GQF2(KB, VB, 8);             \
    else GQF2(KB, VB, 4);                  \
  } while (0)
    if (d <= 64 && dv <= 64) GQF(4, 4);
    else if (d <= 64 && dv <= 128) GQF(4, 8);
    else if (d <= 128 && dv <= 64) GQF(8, 4);
    else GQF(8, 8);
#undef GQF
#undef GQF2
    return (int)hipGetLastError();
  }
  int KT = 64;
  if (gqa_lds(d, dv, KT) > 150 * 1024) KT = 32;
  const long lds = gqa_lds(d, dv, KT);
  if (lds > 150 * 1024) return -2;
  const int R = H / G;
  const dim3 grid(n_tiles, G, (R + GA_ROWS - 1) / GA_ROWS);
  const int nj = (dv + 63) / 64;
  const int TQ = dllm_gqa_tile_tokens(H, G, 0);
  if (f32)
    return launch_gqa_t<float>(nj, grid, lds, st, q, kc, vc, bt, bt_ld, BSZ, qstart, qlen, ctx, tile_seq, tile_tok0, gate, ldg,
                               out, H, G, d, dv, TQ, KT, win, GV, out32, keep, sink, chunk, cap, sinks, ldo, slopes, ghead);
  return launch_gqa_t<u16>(nj, grid, lds, st, q, kc, vc, bt, bt_ld, BSZ, qstart, qlen, ctx, tile_seq, tile_tok0, gate, ldg, out,
                           H, G, d, dv, TQ, KT, win, GV, out32, keep, sink, chunk, cap, sinks, ldo, slopes, ghead);
}

extern "C" int dllm_qk_norm_prep(const void* proj, long ld, int f32, const float* bias, int H, int G, int M, int d, int dv,
                                 const float* qw, const float* kw, const float* cos_sin, int tab_w, int rot, float eps,
                                 float qscale, const int* pos, const int* slots, void* kc, void* vc, void* q, long T, int BSZ,
                                 void* zero_rows, int zw, hipStream_t st) {
  if (T <= 0) return 0;
  if (rot < 0 || rot > d || (rot & 1) || rot > tab_w || H < 1 || G < 1 || H % G || M < 1) return -1;
  const int units = H * M + (kc ? G * M : 0);
  const dim3 grid((unsigned)T, (units + 3) / 4);
  if (f32)
    hipLaunchKernelGGL(qk_norm_prep_kernel<float>, grid, dim3(256), 0, st, (const float*)proj, ld, bias, H, G, M, d, dv, qw, kw,
                       cos_sin, tab_w, rot, eps, qscale, pos, slots, (float*)kc, (float*)vc, (float*)q, BSZ, (uint32_t*)zero_rows, zw);
  else
    hipLaunchKernelGGL(qk_norm_prep_kernel<u16>, grid, dim3(256), 0, st, (const u16*)proj, ld, bias, H, G, M, d, dv, qw, kw,
                       cos_sin, tab_w, rot, eps, qscale, pos, slots, (u16*)kc, (u16*)vc, (u16*)q, BSZ, (uint32_t*)zero_rows, zw);
  return (int)hipGetLastError();
}

extern "C" int dllm_diff_combine(const float* a, void* out, int f32, long T, int H, int G, int dv, float lam, float eps,
                                 float scale, hipStream_t st) {
  if (T <= 0) return 0;
  if (H < 1 || G < 1 || H % G) return -1;
  const long units = T * H;
  const dim3 grid((unsigned)((units + 3) / 4));
  if (f32)
    hipLaunchKernelGGL(diff_combine_kernel<float>, grid, dim3(256), 0, st, a, (float*)out, units, H, G, dv, lam, eps, scale);
  else
    hipLaunchKernelGGL(diff_combine_kernel<u16>, grid, dim3(256), 0, st, a, (u16*)out, units, H, G, dv, lam, eps, scale);
  return (int)hipGetLastError();
}

extern "C" int dllm_proj_norm_prep(const void* proj, long ld, int f32, int H, int G, int d, int dv, const float* qw,
                                   const float* kw, const float* cos_sin, int tab_w, int rot, int inter, float eps,
                                   const float* qscale, int vnorm, const int* pos, const int* slots, void* kc, void* vc, void* q,
                                   long T, int BSZ, void* zrow, int zn, hipStream_t st) {
  if (T <= 0) return 0;
  if (rot < 0 || rot > d || (rot & 1) || rot > tab_w || H < 1 || G < 1 || H % G) return -1;
  const dim3 grid((unsigned)T);
  if (f32)
    hipLaunchKernelGGL(proj_norm_prep_kernel<float>, grid, dim3(256), 0, st, (const float*)proj, ld, H, G, d, dv, qw, kw, cos_sin,
                       tab_w, rot, inter, eps, qscale, vnorm, pos, slots, (float*)kc, (float*)vc, (float*)q, BSZ, (float*)zrow, zn);
  else
    hipLaunchKernelGGL(proj_norm_prep_kernel<u16>, grid, dim3(256), 0, st, (const u16*)proj, ld, H, G, d, dv, qw, kw, cos_sin,
                       tab_w, rot, inter, eps, qscale, vnorm, pos, slots, (u16*)kc, (u16*)vc, (u16*)q, BSZ, (u16*)zrow, zn);
  return (int)hipGetLastError();
}

extern "C" int dllm_rope_prep(const void* proj, long ld, int f32, int H, int G, int d, int dv, const float* cos_sin, int tab_w,
                              int rot, float qscale, const int* pos, const int* slots, void* kc, void* vc, void* q, long T,
                              int BSZ, int ucol, int ff, void* act, long lda, void* zrow, long ldz, int zn,
                              const float* bias, const float* qtab, hipStream_t st) {
  if (T <= 0) return 0;
  if (rot < 0 || rot > d || (rot & 1) || rot > tab_w || H < 1 || G < 1 || H % G || (act && ff < 1)) return -1;
  const dim3 grid((unsigned)T, (H + G + 3) / 4);
  // 16-byte vectors for the activation: every row start and the row length are multiples of 8 entries
  const int vec = act && !f32 && ff % 8 == 0 && ucol % 8 == 0 && ld % 8 == 0 && lda % 8 == 0 && (uintptr_t)proj % 16 == 0 &&
                  (uintptr_t)act % 16 == 0;
  if (f32)
    hipLaunchKernelGGL(rope_prep_kernel<float>, grid, dim3(256), 0, st, (const float*)proj, ld, H, G, d, dv, cos_sin, tab_w, rot,
                       qscale, pos, slots, (float*)kc, (float*)vc, (float*)q, BSZ, ucol, ff, (float*)act, lda, vec, (float*)zrow,
                       ldz, zn, bias, qtab);
  else
    hipLaunchKernelGGL(rope_prep_kernel<u16>, grid, dim3(256), 0, st, (const u16*)proj, ld, H, G, d, dv, cos_sin, tab_w, rot,
                       qscale, pos, slots, (u16*)kc, (u16*)vc, (u16*)q, BSZ, ucol, ff, (u16*)act, lda, vec, (u16*)zrow, ldz, zn,
                       bias, qtab);
  return (int)hipGetLastError();
}
