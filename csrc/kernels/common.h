// Shared device helpers for the gfx950 (CDNA4) kernel library.
//
// Conventions used by every kernel in csrc/kernels:
//   * wave = 64 lanes; block sizes are multiples of 64;
//   * bf16 tensors are moved as 16-byte vectors (8 x bf16) — hipcc does not vectorise
//     scalar bf16 loads (cdna_hip_programming.md Guideline 13);
//   * accumulation in f32; bf16 rounding is round-to-nearest-even.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint16_t u16;

struct __attribute__((aligned(16))) u16x8 { u16 v[8]; };
struct __attribute__((aligned(8))) u16x4 { u16 v[4]; };

static __device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float(((uint32_t)h) << 16); }

// Round to nearest even by the conversion instruction: bit for bit what a rounding by hand in seven integer operations gives, over all
// 2^32 floats (NaN stays NaN, a signalling one becomes quiet).  A 256 x 256 output tile rounds 65536 values two or three times while
// nothing else runs on its CU: TinyLlama's prompts 1.05x whole, a batch of encoded queries 572 -> 507 us.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
static __device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
static __device__ __forceinline__ u16 f2bf(float f) { return __builtin_bit_cast(u16, (__bf16)f); }

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ uint4 ld16(const void* p) { return *reinterpret_cast<const uint4*>(p); }
// non-temporal 16-B load (streamed-once operands: decode weights) -> bf16x8 operand
static __device__ __forceinline__ bf16x8 ldnt_bf16x8(const void* p) {
  return __builtin_bit_cast(bf16x8, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)));
}
static __device__ __forceinline__ void st16(void* p, uint4 v) { *reinterpret_cast<uint4*>(p) = v; }

// ---- in-launch hand-off helpers (cdna_hip_programming.md Guideline 16, recipe R1):
// payload stored WRITE-THROUGH (sc1, 16 B) so no release fence (which writes back the whole XCD
// L2) is needed; every storing wave drains with s_waitcnt vmcnt(0) before the workgroup barrier;
// one lane takes the ticket with a relaxed agent-scope atomic; the consumer reads the payload
// ONLY with sc1 loads (bypass its L1), so it needs no acquire fence either.
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}
static __device__ __forceinline__ void st_wt16(__amdgpu_buffer_rsrc_t r, unsigned byte_off, float4 v) {
  const u32x4 u = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
  __builtin_amdgcn_raw_buffer_store_b128(u, r, byte_off, 0, 16 /* sc1 */);
}
static __device__ __forceinline__ float4 ld_wt16(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
  const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 16 /* sc1 */);
  return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
}
// Drain this wave's stores, barrier, one ticket per workgroup; returns true in the LAST arriver.
// `flag` must be a __shared__ int.  The counter is re-armed (0) by the last arriver.
static __device__ __forceinline__ bool ticket_last(int* counter, int expected, int* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = (old == expected - 1);
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  return *flag != 0;
}

// unpack 8 bf16 (one uint4) to f32
static __device__ __forceinline__ void unpack8(uint4 v, float* f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(w[i] << 16);
    f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

static __device__ __forceinline__ uint4 pack8(const float* f) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = f2bf2(f[2 * i], f[2 * i + 1]);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Exchanges across a wave for constant distances, all lanes active: v of lane ^ O as DPP moves and row swaps, which are vector
// instructions, where __shfl_xor goes through the LDS crossbar (ds_bpermute, an address to compute and a wait).  A wave's sum is six
// of them one behind the other, and a GEMV has as many for each of its outputs: a single chat turn on TinyLlama (57 tokens in, 16 out)
// 12.3 -> 11.7 ms, the mixture's batch of 12 (router, norms, attention) 7.25 -> 7.0.
template <class T> static __device__ __forceinline__ T lane_xor(T v, const int o) {
  static_assert(sizeof(T) == 4, "a register a lane");
  const int u = __builtin_bit_cast(int, v);
  int r;
  if (o == 1) r = __builtin_amdgcn_mov_dpp(u, 0xB1, 0xf, 0xf, true);              // quad_perm 1 0 3 2
  else if (o == 2) r = __builtin_amdgcn_mov_dpp(u, 0x4E, 0xf, 0xf, true);         // quad_perm 2 3 0 1
  else if (o == 4) r = __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(u, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);  // ^7, ^3
  else if (o == 8) r = __builtin_amdgcn_mov_dpp(u, 0x128, 0xf, 0xf, true);        // row_ror 8
  else if (o == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);   // even rows twice, odd rows twice
    r = (int)(__lane_id() & 16 ? s[0] : s[1]);
  } else {
    const auto s = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);   // the lower half twice, the upper twice
    r = (int)(__lane_id() & 32 ? s[0] : s[1]);
  }
  return __builtin_bit_cast(T, r);
}
// v + lane_xor(v, o), max(v, lane_xor(v, o))
static __device__ __forceinline__ float lane_add(float v, const int o) {
  const unsigned u = __float_as_uint(v);
  if (o == 16) { const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false); return __uint_as_float(s[0]) + __uint_as_float(s[1]); }
  if (o == 32) { const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false); return __uint_as_float(s[0]) + __uint_as_float(s[1]); }
  return v + lane_xor(v, o);
}
static __device__ __forceinline__ float lane_max(float v, const int o) {
  const unsigned u = __float_as_uint(v);
  if (o == 16) { const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false); return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1])); }
  if (o == 32) { const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false); return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1])); }
  return fmaxf(v, lane_xor(v, o));
}

static __device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = lane_add(v, o);
  return v;
}

static __device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = lane_max(v, o);
  return v;
}

// Block-wide sum for blockDim.x <= 1024 (multiple of 64). `red` must hold >= 16 floats.
static __device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

// x (1 + erf(x / sqrt 2)) / 2 for values that end in bf16: max(x, 0) - |x| erfc(|x| / sqrt 2) / 2, with erfc(z) = exp(-z^2) t P(t), t = 1 / (1 + z / 2);
// 2 P: a fit of erfcx(z) / t on z from 0 to 10 to the least largest relative error (4.3e-8, reweighted least squares).  Half of erff's instructions, which
// were most of an epilogue, and no cancellation where 1 + erf is small: the largest relative error against 64 bits is 3e-7 from -1 to 1 and 7e-7 to -3,
// 9e-6 below (with erff 1.4e-7, 7e-6, 4e-2 to -5 and 1), and of the 65280 finite bf16 inputs none whose result is 2^-125 or more rounds to another bf16
// than the exact value (197 with erff; smaller results, at x below -13, may be 0: the exponential's instruction has no subnormal numbers).  3571 x 1536 x 384 with it: 16.0 us, with erff 16.9.  NaN and infinities as there (-inf: NaN).
static __device__ __forceinline__ float gelu_bf(float x) {
  const float t = __builtin_amdgcn_rcpf(fmaf(fabsf(x), 0.35355339059327373f, 1.f)), u = x * 0.84932180028801907f;      // sqrt(log2(e) / 2)
  float p = fmaf(t, -0.029534505680203438f, 0.14228759706020355f);
  p = fmaf(t, p, -0.24360017478466034f);
  p = fmaf(t, p, 0.13903383910655975f);
  p = fmaf(t, p, -0.013312997296452522f);
  p = fmaf(t, p, 0.10134349763393402f);
  p = fmaf(t, p, 0.12155186384916306f);
  p = fmaf(t, p, 0.1411876529455185f);
  p = fmaf(t, p, 0.14104321599006653f);
  const float q = t * p * __builtin_amdgcn_exp2f(-u * u);
  return fmaf(-fmaxf(-x, fminf(x, 16.f)), q, fmaxf(x, 0.f));
}
