// What the tiled GEMMs (tgemm.hip, wide_gemm.hip) share.
#pragma once
#include "common.h"
#include "tgemm_args.h"

namespace dllm {
// wide_gemm.hip: the 256 x 256 tile of four waves
int wide_gemm(const GemmArgs& a, int epi, hipStream_t st);

// Copy-out of a QKV tile whose row-scaled, rounded outputs lie in LDS (so [BM][OLD]), a workgroup of NT threads: q and k rotated in row
// vectors of eight pairs, q to q_out, k to its pages, V to rows or to the V^T pages.  s_slot / s_pos [BM]: cache slot and position of
// each row; s_run [BM]: scratch (0 alone, 1 in a run, 2 a run's first).  (Rotated in registers every lane waited for the table rows of
// its output rows one after the other, and V went out in 2-byte stores 32 B apart: of a 256 x 128 tile's 54 us at 2100 rows that was 21.)
template <int BM, int BN, int OLD, int NT>
__device__ __forceinline__ void qkv_copy_out(const GemmArgs& a, const u16* so, const int* s_slot, const int* s_pos, int* s_run, const int M,
                                             const int m0, const int n0) {
  const int N = a.N, d = a.d, hd = d / 2, nq = a.nq, nkv = a.nkv;
  const int qcols = nq * d, kcols = nkv * d, vcol0 = qcols + kcols;
  for (int e = threadIdx.x; e < BM * (BN / 16); e += NT) {
    const int rl = e / (BN / 16), u = e % (BN / 16), c0 = 32 * (u >> 1) + 8 * (u & 1);
    const int m = m0 + rl, n = n0 + c0;
    if (m >= M || n >= vcol0 || n >= N) continue;
    const bool isq = n < qcols;
    const int cc = isq ? n : n - qcols, head = cc / d, o = cc % d, d1 = 16 * (o >> 5) + (o & 15);
    const float* cs = a.cos_sin + (long)s_pos[rl] * d + d1;
    float co[8], si[8], x1[8], x2[8], r1[8], r2[8];
    *(float4*)&co[0] = *(const float4*)cs;
    *(float4*)&co[4] = *(const float4*)(cs + 4);
    *(float4*)&si[0] = *(const float4*)(cs + hd);
    *(float4*)&si[4] = *(const float4*)(cs + hd + 4);
    unpack8(*reinterpret_cast<const uint4*>(so + rl * OLD + c0), x1);
    unpack8(*reinterpret_cast<const uint4*>(so + rl * OLD + c0 + 16), x2);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      r1[j] = x1[j] * co[j] - x2[j] * si[j];
      r2[j] = x2[j] * co[j] + x1[j] * si[j];
    }
    const int slot = s_slot[rl];
    u16* dst = isq ? a.q_out + ((long)m * nq + head) * d
                   : (slot >= 0 ? a.kc + (((long)(slot >> 4) * nkv + head) * 16 + (slot & 15)) * d : nullptr);
    if (dst) {
      st16(dst + d1, pack8(r1));
      st16(dst + hd + d1, pack8(r2));
    }
  }
  if (n0 + BN <= vcol0) return;      // (block-uniform)
  const int v0 = max(0, vcol0 - n0), nv = min(BN, N - n0) - v0;      // this tile's V columns
  if (a.v_rows != nullptr) {
    for (int e = threadIdx.x; e < BM * (nv / 8); e += NT) {
      const int rl = e / (nv / 8), c = v0 + (e % (nv / 8)) * 8;
      if (m0 + rl < M) st16(a.v_rows + (long)(m0 + rl) * a.v_ld + (n0 + c - vcol0), *reinterpret_cast<const uint4*>(so + rl * OLD + c));
    }
    return;
  }
  // V^T cache [block][head][dim][16]: eight rows in eight consecutive slots of half a block (a prompt's) are one 16-byte store per
  // dim, written by the first of them; rows outside such a run store their two bytes.  Rows and columns by the tile's constants: divisions
  // by the tile's number of V columns and by d made a decode step's tiles slower than stores from registers (96 rows, 6144 columns
  // of 128: 25.5 from registers, 27.9, here 25.7 us)
  for (int r = threadIdx.x; r < BM; r += NT) {
    const int sl = s_slot[r], st = r - (sl & 7);
    bool run = sl >= 0 && st >= 0 && st + 7 < BM && m0 + st + 7 < M;
    if (run)
      for (int j = 0; j < 8; ++j) run = run && s_slot[st + j] == (sl & ~7) + j;
    s_run[r] = run ? 1 + (st == r) : 0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < BM * BN; e += NT) {
    const int rl = e / BN, c = e % BN;
    if (c < v0 || c >= v0 + nv || m0 + rl >= M) continue;
    const int run = s_run[rl], slot = s_slot[rl];
    if (slot < 0 || run == 1) continue;
    u16* vo = a.vc + ((long)(slot >> 4) * nkv * d + (n0 + c - vcol0)) * 16 + (slot & 15);      // (head, dim: the column itself)
    if (run == 2) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        w[j] = (uint32_t)so[(rl + 2 * j) * OLD + c] | ((uint32_t)so[(rl + 2 * j + 1) * OLD + c] << 16);
      st16(vo, make_uint4(w[0], w[1], w[2], w[3]));
    } else *vo = so[rl * OLD + c];
  }
}
}  // namespace dllm
