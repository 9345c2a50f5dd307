// Chunks of a packed batch: sequence s has ceil(qlen[s] / L) chunks, numbered over all sequences in order.
#pragma once
#include <hip/hip_runtime.h>

namespace dllm {

// inclusive sum over the lanes of a wave
static __device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o);
    if (lane >= o) v += u;
  }
  return v;
}

// chunk number `flat` -> its sequence and its place there; false past the last one (the same for the whole workgroup)
template <int L> static __device__ __forceinline__ bool find_chunk(const int* qlen, int S, int flat, int& s, int& c) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int i0 = 0; i0 < S; i0 += 64) {
    const int n = i0 + lane < S ? (max(qlen[i0 + lane], 0) + L - 1) / L : 0;
    const int up = wave_scan(n, lane);
    const unsigned long long m = __ballot(base + up > flat);
    if (m) {
      const int l = __ffsll(m) - 1;
      s = i0 + l;
      c = flat - base - (__shfl(up, l) - __shfl(n, l));
      return true;
    }
    base += __shfl(up, 63);
  }
  return false;
}

// chunks of the sequences before s (every lane of the wave calls it)
template <int L> static __device__ __forceinline__ int chunks_before(const int* qlen, int s) {
  int n = 0;
  for (int i = threadIdx.x & 63; i < s; i += 64) n += (max(qlen[i], 0) + L - 1) / L;
#pragma unroll
  for (int o = 32; o; o >>= 1) n += __shfl_xor(n, o);
  return n;
}

// Clear the rows of `out` that belong to no sequence (the tokens a captured step is padded with): a wave asks for one row at a
// time and writes only those.  part of parts: this workgroup's share, `waves` waves a workgroup.
template <typename T>
static __device__ __forceinline__ void zero_free_rows(T* out, long rows, int width, const int* qstart, const int* qlen, int S, long part,
                                                      long parts, int waves) {
  const int lane = threadIdx.x & 63;
  for (long r = part * waves + (threadIdx.x >> 6); r < rows; r += parts * waves) {
    bool in = false;
    for (int s0 = lane; s0 < S; s0 += 256) {      // four sequences a lane in flight: a batch's slots cost one round trip
      int a[4], n[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] = qstart[min(s0 + 64 * u, S - 1)];
        n[u] = qlen[min(s0 + 64 * u, S - 1)];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) in |= r >= a[u] && r < (long)a[u] + n[u];
    }
    if (__ballot(in)) continue;
    for (int c = lane; c < width; c += 64) out[r * width + c] = T(0);
  }
}

}  // namespace dllm
