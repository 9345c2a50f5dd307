// Chunk-parallel selective scan (Mamba-1) for prompt portions (gfx950, wave64); decode steps and short portions run the
// token-by-token kernel of seqmix.hip.  Per channel and state
//
//     S_t = exp(dt_t A) S_(t-1) + dt_t x_t B_t,   y_t = sum_n S_t C_t + D x_t,   out = y silu(z)
//
// With chunks of 32 tokens: scan_sum runs every chunk from a zero state and keeps its end and the sum of its steps
// (the chunk's decay is exp(A sum dt)); scan_carry walks the chunks, one multiply-add per state; scan_out runs every
// chunk again from its true start and writes the outputs.  A thread has one channel with all its states in
// registers: no sums across lanes, B and C rows are broadcast from LDS, and the 64 channels of a wave read and write
// whole rows.  All of it in f32.
//
// What bounds it: the exponentials, one per token, channel and state in either pass (4001 tokens x 2048 channels x 16
// states: 131M, 14 us of the transcendental unit a pass) and the 20 plain instructions a token and state around them.
// One sequence of 4096 tokens there: sums 43, carry 21, outputs 55 us; token by token 128 workgroups take 884 us.
#include "chunks.h"
#include "common.h"

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <typename T> __device__ __forceinline__ void stf(T* p, float v);
template <> __device__ __forceinline__ void stf<u16>(u16* p, float v) { *p = f2bf(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }
// exp(dt A): bf16 models on the hardware's exponential, as in the token-by-token kernel, with log2 e in A
template <typename T> struct Decay;
template <> struct Decay<u16> {
  static __device__ __forceinline__ float pre(float a) { return a * 1.44269504088896f; }
  static __device__ __forceinline__ float f(float x) { return __builtin_amdgcn_exp2f(x); }
};
template <> struct Decay<float> {
  static __device__ __forceinline__ float pre(float a) { return a; }
  static __device__ __forceinline__ float f(float x) { return expf(x); }
};

// log(1 + e^x) = max(x, 0) + log1p(u), u = e^-|x|, log1p(u) = 2 atanh(z), z = u / (2 + u) <= 1 / 3, as its power series; the divisor's
// rounding, the quotient's remainder and the rounding of the last sum are carried.  Root mean square error against 64 bits in units of
// 2^-24 (log1pf(expf(x)) in brackets; 4M points a range): -20 .. -5 0.59 (0.59), -5 .. -1 0.60 (0.60), -1 .. 0 0.54 (0.54), 0 .. 1
// 0.46 (0.52), 1 .. 5 0.43 (0.46), 5 .. 20 0.34 (0.34).  The chunk kernels on 4096 tokens: 112 us against 142 with log1pf.
__device__ __forceinline__ float softplus_f(float x) {
  const float u = expf(-fabsf(x)), d = 2.f + u, dl = u - (d - 2.f), r = __builtin_amdgcn_rcpf(d);
  float z = u * r;
  z = fmaf(fmaf(-z, dl, fmaf(-z, d, u)), r, z);
  const float zl = fmaf(-z, dl, fmaf(-z, d, u)) * r, w = z * z, z2 = 2.f * z;
  float p = fmaf(w, 1.f / 15.f, 1.f / 13.f);
  p = fmaf(w, p, 1.f / 11.f);
  p = fmaf(w, p, 1.f / 9.f);
  p = fmaf(w, p, 1.f / 7.f);
  p = fmaf(w, p, 1.f / 5.f);
  p = fmaf(w, p, 1.f / 3.f);
  const float y = fmaf(z2 * w, p, 2.f * zl);
  if (!(x > 0.f)) return z2 + y;
  const float s = x + z2, b = s - x, e = (x - (s - b)) + (z2 - b);      // x + z2 = s + e
  return x > 1e30f ? x : s + (e + y);
}

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }

constexpr int SC_L = 32;      // tokens per chunk
constexpr int SC_AHEAD = 8;   // tokens whose inputs are in flight
constexpr long SC_SCRATCH = 1L << 26;     // entries of chunk ends (256 MB) up to which all channels go at once; else some at a time: 2048
                                          // channels of 16 states from 61000 tokens on

template <typename T> struct MambaArgs {
  const T *xc, *dt_raw, *dbc, *xz;
  long ldd, ldz;
  int dt_rank;
  const float *dt_bias, *A, *D;
  float* ssm;
  T* conv;
  int Km1;
  const int *qstart, *qlen, *ctx, *rows;
  T* out;
  int S, C, N, nchunks;
  int c0, CC;               // first channel of the launch, channels that the scratch holds
  float *ends, *steps;      // [chunks][N][CC], [chunks][CC]
  long tokens;
};

// OUT = false: scan_sum, true: scan_out.  NP >= N states in registers (the padded ones stay zero).
template <typename T, int NP, bool OUT>
__global__ void __launch_bounds__(256) scan_chunk_kernel(MambaArgs<T> a) {
  constexpr int W = OUT ? 2 * NP : NP;      // staged numbers per token: B (and C)
  __shared__ __attribute__((aligned(16))) float bc[SC_L * W];
  int s, ch;
  if (!dllm::find_chunk<SC_L>(a.qlen, a.S, blockIdx.y, s, ch)) return;
  const int n = a.qlen[s], t0 = ch * SC_L, nt = min(SC_L, n - t0), p0 = a.ctx[s] - n;
  const long tok0 = a.qstart[s] + t0;
  for (int e = threadIdx.x; e < SC_L * W; e += 256) {
    const int t = e / W, k = e % W, i = k < NP ? k : k - NP;
    bc[e] = t < nt && i < a.N ? ldf(a.dbc + (tok0 + t) * a.ldd + a.dt_rank + (k < NP ? 0 : a.N) + i) : 0.f;
  }
  __syncthreads();
  const int cc = blockIdx.x * 256 + threadIdx.x, c = a.c0 + cc;
  if (cc >= a.CC || c >= a.C) return;
  float A[NP], S[NP];
  float* ends = a.ends + (long)blockIdx.y * a.N * a.CC + cc;
  const bool carried = OUT && (ch > 0 || p0 > 0);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    A[i] = i < a.N ? Decay<T>::pre(a.A[(long)c * a.N + i]) : 0.f;
    S[i] = carried && i < a.N ? ends[(long)i * a.CC] : 0.f;
  }
  const float dtb = a.dt_bias[c], skip = OUT ? a.D[c] : 0.f;
  float sum = 0.f;
  auto group = [&](int u0, int m) {      // tokens u0 .. u0 + m - 1 of the chunk; m is SC_AHEAD but for the last group
    float raw[SC_AHEAD], x[SC_AHEAD], z[SC_AHEAD];
#pragma unroll
    for (int j = 0; j < SC_AHEAD; ++j) {
      const long tok = tok0 + u0 + min(j, m - 1);
      raw[j] = ldf(a.dt_raw + tok * a.C + c);
      x[j] = ldf(a.xc + tok * a.C + c);
      z[j] = OUT ? ldf(a.xz + tok * a.ldz + a.C + c) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < SC_AHEAD; ++j) {
      if (j >= m) break;
      const float dt = softplus_f(raw[j] + dtb), dx = dt * x[j];
      const float4* b4 = reinterpret_cast<const float4*>(bc + (u0 + j) * W);
      float y = 0.f;
#pragma unroll
      for (int i = 0; i < NP; i += 4) {
        const float4 b = b4[i / 4];
        const float bv[4] = {b.x, b.y, b.z, b.w};
        const float4 cc = OUT ? b4[(NP + i) / 4] : make_float4(0.f, 0.f, 0.f, 0.f);
        const float cv[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          S[i + k] = Decay<T>::f(dt * A[i + k]) * S[i + k] + dx * bv[k];
          if (OUT) y += S[i + k] * cv[k];
        }
      }
      if (OUT) stf(a.out + (tok0 + u0 + j) * a.C + c, (y + skip * x[j]) * silu_f(z[j]));
      else sum += dt;
    }
  };
  int u0 = 0;
  for (; u0 + SC_AHEAD <= nt; u0 += SC_AHEAD) group(u0, SC_AHEAD);
  if (u0 < nt) group(u0, nt - u0);
  if constexpr (!OUT) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (i < a.N) ends[(long)i * a.CC] = S[i];
    a.steps[(long)blockIdx.y * a.CC + cc] = sum;
  } else if (t0 + nt == n && a.Km1 > 0) {
    // the last K-1 inputs of the sequence: new tokens where there are enough, else the slot's older ones
    T* cs = a.conv + (long)a.rows[s] * a.Km1 * a.C + c;
    const long q0 = a.qstart[s];
    float u[8];
    for (int k = 0; k < a.Km1; ++k) {
      const int i = n - a.Km1 + k;
      u[k] = i >= 0 ? ldf(a.xz + (q0 + i) * a.ldz + c) : (p0 > 0 ? ldf(cs + (long)(a.Km1 + i) * a.C) : 0.f);
    }
    for (int k = 0; k < a.Km1; ++k) stf(cs + (long)k * a.C, u[k]);
  }
}

// chunk ends -> the state before every chunk, in place, and the state behind the last one into the slot
template <typename T> __global__ void __launch_bounds__(256) scan_carry_kernel(MambaArgs<T> a) {
  constexpr int AHEAD = 8;
  const int s = blockIdx.z, i = blockIdx.y;
  const int n = a.qlen[s];
  if (n <= 0) return;
  const int first = dllm::chunks_before<SC_L>(a.qlen, s);
  const int nc = min((n + SC_L - 1) / SC_L, a.nchunks - first);
  const int cc = blockIdx.x * 256 + threadIdx.x, c = a.c0 + cc;
  if (cc >= a.CC || c >= a.C) return;
  float* st = a.ssm + ((long)a.rows[s] * a.C + c) * a.N + i;
  float* u = a.ends + ((long)first * a.N + i) * a.CC + cc;
  const float* d = a.steps + (long)first * a.CC + cc;
  const float A = a.A[(long)c * a.N + i];
  float S = a.ctx[s] - n > 0 ? *st : 0.f;
  for (int c0 = 0; c0 < nc; c0 += AHEAD) {
    float x[AHEAD], g[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const long k = min(c0 + j, nc - 1);
      x[j] = u[k * a.N * a.CC];
      g[j] = d[k * a.CC];
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      if (c0 + j >= nc) break;
      u[(long)(c0 + j) * a.N * a.CC] = S;
      S = expf(A * g[j]) * S + x[j];
    }
  }
  *st = S;
}

// Decode steps: a thread per channel walks its sequence's few new tokens with all states in registers.  What bounds it is the
// chain metadata -> state -> store, so every load of the first token is in flight at once and a workgroup is one wave (768 of
// them for 24 sequences of 2048 channels).  24 sequences of 2048 channels of 16 states: 6.9 us (12.6 MB read and written, 1.8 us of
// it the launch) against 14.0 with 16 lanes a channel, which needs four times the workgroups and sums across lanes.
template <typename T, int NP> __global__ void __launch_bounds__(64) scan_step_kernel(MambaArgs<T> a) {
  __shared__ __attribute__((aligned(16))) float bc[2 * NP];
  const int s = blockIdx.y, lane = threadIdx.x;
  if (s == a.S) {      // one more row of workgroups clears the rows of no sequence
    dllm::zero_free_rows(a.out, a.tokens, a.C, a.qstart, a.qlen, a.S, blockIdx.x, gridDim.x, 1);
    return;
  }
  const int n = a.qlen[s];
  if (n <= 0) return;
  const int c0 = blockIdx.x * 64 + lane, c = c0 < a.C ? c0 : a.C - 1;   // lanes past the last channel shadow it and store nothing
  const bool live = c0 < a.C, carried = a.ctx[s] - n > 0;
  const long q0 = a.qstart[s], slot = a.rows[s];
  float* sp = a.ssm + (slot * a.C + c) * a.N;
  const float* ap = a.A + (long)c * a.N;
  f32x4 A[NP / 4], S[NP / 4];
#pragma unroll
  for (int i = 0; i < NP / 4; ++i) {   // N is a multiple of 4; places past it are read at 0 and made zero
    A[i] = *reinterpret_cast<const f32x4*>(ap + (4 * i < a.N ? 4 * i : 0));
    S[i] = *reinterpret_cast<const f32x4*>(sp + (4 * i < a.N ? 4 * i : 0));
  }
  const float dtb = a.dt_bias[c], skip = a.D[c];
  T* cs = a.conv + slot * a.Km1 * a.C + c;
  T cv[8];   // the last Km1 inputs of the sequence: new tokens where there are enough, else the slot's older ones
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (k < a.Km1) {
      const int i = n - a.Km1 + k;
      cv[k] = i >= 0 ? a.xz[(q0 + i) * a.ldz + c] : cs[(long)(a.Km1 + i) * a.C];
      if (i < 0 && !carried) cv[k] = T(0);
    }
#pragma unroll
  for (int i = 0; i < NP / 4; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      A[i][k] = 4 * i < a.N ? Decay<T>::pre(A[i][k]) : 0.f;
      S[i][k] = carried && 4 * i < a.N ? S[i][k] : 0.f;
    }
  for (int t = 0; t < n; ++t) {
    const long tok = q0 + t;
    const T* bp = a.dbc + tok * a.ldd + a.dt_rank;
    const float raw = ldf(a.dt_raw + tok * a.C + c), x = ldf(a.xc + tok * a.C + c), z = ldf(a.xz + tok * a.ldz + a.C + c);
    __syncthreads();   // the previous token's rows are consumed
    if (lane < 2 * NP) {
      const int i = lane < NP ? lane : lane - NP;
      bc[lane] = i < a.N ? ldf(bp + (lane < NP ? 0 : a.N) + i) : 0.f;
    }
    __syncthreads();
    const float dt = softplus_f(raw + dtb), dx = dt * x;
    float y = 0.f;
#pragma unroll
    for (int i = 0; i < NP / 4; ++i) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(bc + 4 * i), g = *reinterpret_cast<const f32x4*>(bc + NP + 4 * i);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        S[i][k] = Decay<T>::f(dt * A[i][k]) * S[i][k] + dx * b[k];
        y += S[i][k] * g[k];
      }
    }
    if (live) stf(a.out + tok * a.C + c, (y + skip * x) * silu_f(z));
  }
  if (!live) return;
#pragma unroll
  for (int i = 0; i < NP / 4; ++i)
    if (4 * i < a.N) *reinterpret_cast<f32x4*>(sp + 4 * i) = S[i];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (k < a.Km1) cs[(long)k * a.C] = cv[k];
}

template <typename T, int NP> void launch(MambaArgs<T> a, hipStream_t st) {
  for (a.c0 = 0; a.c0 < a.C; a.c0 += a.CC) {      // the stream keeps one group's launches ahead of the next's writes
    const int n = ((a.CC < a.C - a.c0 ? a.CC : a.C - a.c0) + 255) / 256;
    const dim3 g(n, a.nchunks), b(256);
    hipLaunchKernelGGL((scan_chunk_kernel<T, NP, false>), g, b, 0, st, a);
    hipLaunchKernelGGL(scan_carry_kernel<T>, dim3(n, a.N, a.S), b, 0, st, a);
    hipLaunchKernelGGL((scan_chunk_kernel<T, NP, true>), g, b, 0, st, a);
  }
}

int channels_at_once(long nchunks, int C, int N) {
  const long n = SC_SCRATCH / (nchunks * (N + 1L)) / 256 * 256;
  return n < 256 ? (C < 256 ? C : 256) : n < C ? (int)n : C;
}

template <typename T>
int run(const void* xc, const void* dt_raw, const float* dt_bias, const float* A, const void* dbc, long ldd, int dt_rank,
        const float* D, const void* xz, long ldz, float* ssm, void* conv, int Km1, const int* qstart, const int* qlen,
        const int* ctx, const int* rows, void* out, int S, long tokens, int C, int N, float* scratch, hipStream_t st) {
  MambaArgs<T> a{(const T*)xc, (const T*)dt_raw, (const T*)dbc, (const T*)xz, ldd, ldz, dt_rank, dt_bias, A, D, ssm, (T*)conv,
                 Km1, qstart, qlen, ctx, rows, (T*)out, S, C, N, (int)(tokens / SC_L) + S, 0, C, scratch, nullptr, tokens};
  if (!scratch) {
    const dim3 g((C + 63) / 64, S + 1);
    if (N <= 8) hipLaunchKernelGGL((scan_step_kernel<T, 8>), g, dim3(64), 0, st, a);
    else if (N <= 16) hipLaunchKernelGGL((scan_step_kernel<T, 16>), g, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((scan_step_kernel<T, 32>), g, dim3(64), 0, st, a);
    return (int)hipGetLastError();
  }
  a.CC = channels_at_once(a.nchunks, C, N);
  a.steps = scratch + (long)a.nchunks * N * a.CC;
  if (a.nchunks > 65535) return -3;
  if (N <= 8) launch<T, 8>(a, st);
  else if (N <= 16) launch<T, 16>(a, st);
  else launch<T, 32>(a, st);
  return (int)hipGetLastError();
}

}  // namespace

// f32 entries of scratch for a step of T tokens and S sequences; 0: not taken (more states than a thread keeps, or more
// chunks than a grid's second dimension)
extern "C" long dllm_scan_chunks_scratch(long T, int S, int C, int N) {
  const long nc = T / SC_L + S;
  return N < 1 || N > 32 || nc < 1 || nc > 65535 ? 0 : nc * channels_at_once(nc, C, N) * (N + 1L);
}

// May the step kernel take it?  Whole, aligned vectors of states.
extern "C" int dllm_scan_step_ok(int N, const void* ssm, const void* A) {
  return N % 4 == 0 && N <= 32 && (((uintptr_t)ssm | (uintptr_t)A) & 15) == 0;
}

// the arguments of dllm_selective_scan, and the scratch; without scratch the step kernel (dllm_scan_step_ok)
extern "C" int dllm_scan_chunks(const void* xc, const void* dt_raw, int f32, const float* dt_bias, const float* A, const void* dbc,
                                long ldd, int dt_rank, const float* D, const void* xz, long ldz, float* ssm, void* conv, int Km1,
                                const int* qstart, const int* qlen, const int* ctx, const int* rows, void* out, int S, long T,
                                int C, int N, float* scratch, hipStream_t st) {
  if (S <= 0 || T <= 0) return 0;
  if (N < 1 || N > 32 || Km1 < 0 || Km1 > 8) return -1;
  return f32 ? run<float>(xc, dt_raw, dt_bias, A, dbc, ldd, dt_rank, D, xz, ldz, ssm, conv, Km1, qstart, qlen, ctx, rows, out, S, T,
                          C, N, scratch, st)
             : run<u16>(xc, dt_raw, dt_bias, A, dbc, ldd, dt_rank, D, xz, ldz, ssm, conv, Km1, qstart, qlen, ctx, rows, out, S, T,
                        C, N, scratch, st);
}
