// Decode GEMM on fragment-major weights:  Y = epilogue(X[M, K] . W[N, K]^T),  M <= 64, bf16 in, f32 accumulate.
//
// What bounds a projection of 4-64 rows is not its weight stream (TinyLlama's Wo at 48 rows: 11.1 us from HBM, 10.2 us with the
// weights in L2) but the rate at which a CU takes in operands that lie in rows: an MFMA fragment is 16 rows x 64 bytes, neighbouring
// lanes read different rows, and a wave's load touches 16 cache lines for the bytes of 8.  So here no load does that:
//   * W is kept as [N / 16][K / 32][64 lanes][8] (ops.gemm.frag_weight): a fragment is 1 KB, contiguous over the lanes;
//   * X is loaded in rows (a quarter of a wave per row and 128 k), goes through a piece of LDS that belongs to the wave alone (no
//     barrier; row pitch 16 bytes off the power of two, so reads and writes meet no bank twice) and comes back as fragments.  Up to
//     16 rows it is read as fragments at once: there the rows of a load are few.
// Each on its own, at 48 rows: 2560 x 2048 10.2 us in rows, 8.9 W, 8.7 X, 7.2 both; 2048 x 5632 14.0, 11.6, 12.7, 10.5; 16 rows
// 6.7, 5.5, 6.2, 5.2 and 10.7, 8.9, 10.1, 8.6 (the rows of W from HBM, plain product, in a captured graph).
//
// A workgroup owns NT 16-column tiles; its VS groups of four waves each take one split of K (so the order of every sum is that of
// skinny_gemm.hip with as many splits: wave order ((w0 + w2) + (w1 + w3)), splits in order), gridDim.y workgroups share a tile
// through write-through slabs and a ticket (2 to 3 us: only where a tile's K is long).  Partial tiles meet in LDS.
//
// Epilogues (those of tgemm.hip, same roundings): PLAIN; RESADD (residual add in place, row sums of squares per tile); QKV (row
// scale, RoPE, q and paged K / V writes); SWIGLU (row scale, silu(g) u).  What an epilogue reads (residual, positions, slots, cos /
// sin) is loaded at the kernel's start.  The row scale of a folded RMSNorm needs no partial sums from the producer: every wave has
// all of its K range of X in fragments, and X . X^T's diagonal, one more MFMA per fragment, is the rows' sums of squares.
// GLU and GELU are the activations of layer-list feed-forwards, on the rounded product as their own launches do them (a launch of its
// own: 3.4 us and the gap before it).  QKV, SWIGLU and GLU weights are stored with the halves of a pair 8 columns apart in one tile (frag_weight).
#include <type_traits>

#include "common.h"

namespace {
enum { DG_PLAIN = 0, DG_RESADD = 1, DG_QKV = 2, DG_SWIGLU = 3, DG_GLU = 4, DG_GELU = 5 };

struct DgArgs {
  const u16* X;
  long ldx;
  const u16* W;
  u16* Y;
  long ldy;
  int M, N, K, kchunk, S;
  float* part;
  int* counters;
  u16* res;           // RESADD: [M, ldr], updated in place
  long ldr;
  float* ssq_out;     // RESADD: per-tile row sums of squares, ssq_out[tile * ssq_ld + m]
  long ssq_ld;
  float scale, eps;   // QKV / SWIGLU: row scale rsqrt(sum x^2 * scale + eps)
  const int* pos;
  const float* cos_sin;
  const int* slots;
  u16* q_out;
  u16* kc;
  u16* vc;
  u16* v_rows;        // V row-major [M, v_ld] instead of the V^T cache
  long v_ld;
  int nq, nkv, d;
  const float* bias;  // GLU: over the gate columns, then the up columns (null: none)
  int mode;           // GLU: 0 silu, 1 clamped, 2 tanh GELU (glu_act of seqmix.hip)
  float limit, alpha;
};

__device__ __forceinline__ uint4 ldb16(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// the loads of a stage stay together, behind the products before them
__device__ __forceinline__ void keep_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int MT, int NT, int VS, int EPI>
struct Dg {
  static constexpr int WV = 4 * VS, T = 64 * WV, NC = 16 * NT, MR = 16 * MT, LD = NC + 4;
  static constexpr bool XL = MT >= 2, SQ = EPI == DG_QKV || EPI == DG_SWIGLU, PAIR = SQ || EPI == DG_GLU;
  // k-steps of 32 in flight per stage (two stages): registers of 16 waves, or of many fragments, hold two
  static constexpr int U = VS == 4 || NT + MT > 4 ? 2 : 4;
  static constexpr int PX = 64 * U + 16;      // bytes of a staged row
  static constexpr int REG = (XL && MR * PX > MR * LD * 4) ? MR * PX : MR * LD * 4;   // a wave's piece of LDS
  static constexpr int ITEMS = MR * NC / (PAIR ? 8 : 4), NI = (ITEMS + T - 1) / T;
  static constexpr int LDS = WV * REG + (SQ ? WV * MR * 4 : MR * (NC / 4) * 4) + 16;
};

// HALVES: a wave's K is that many half stages or fewer (0: any number, two stages at a time).  A step that does not exist is no traffic to
// memory but passes through the caches' pipe like any other: two stages for waves of three steps cost 16 rows of 11264 x 768 in two splits
// 8.2 us for 6.6.  (As ways through one kernel the forms cost it registers, and a fourth of its waves.)
template <int MT, int NT, int VS, int EPI, int HALVES>
__global__ void __launch_bounds__(256 * VS) dgemm_kernel(DgArgs a) {
  using C = Dg<MT, NT, VS, EPI>;
  constexpr int NC = C::NC, MR = C::MR, LD = C::LD, U = C::U, WV = C::WV, T = C::T, NI = C::NI, PX = C::PX;
  constexpr bool XL = C::XL, PAIR = C::PAIR, SQ = C::SQ;
  extern __shared__ __attribute__((aligned(16))) unsigned char dg_smem[];
  float* s_tail = reinterpret_cast<float*>(dg_smem + WV * C::REG);      // row sums: [WV][MR] of X, or [MR][NC / 4] of the result
  int* s_last = reinterpret_cast<int*>(s_tail + (SQ ? WV * MR : MR * (NC / 4)));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wv = wave & 3, grp = wave >> 2;
  const int g = lane >> 4, r16 = lane & 15;
  const int tile = blockIdx.x, split = blockIdx.y * VS + grp, col0 = tile * NC;
  const int M = a.M, N = a.N, K = a.K;
  const int kbeg = min(K, split * a.kchunk), kend = min(K, kbeg + a.kchunk);      // a group past the last split has nothing
  const int kw = (((kend - kbeg + 3) / 4) + 31) & ~31;
  const int wk0 = min(kend, kbeg + wv * kw), wk1 = min(kend, wk0 + kw);

  // ---- what the epilogue reads, first: item i of a thread is row (t + i T) / per row, four columns (or two times four)
  constexpr int IPR = C::ITEMS / MR;      // items per row
  u16x4 e_res[EPI == DG_RESADD ? NI : 1];
  int e_slot[EPI == DG_QKV ? NI : 1], e_pos[EPI == DG_QKV ? NI : 1];
  if constexpr (EPI == DG_RESADD || EPI == DG_QKV) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int it = threadIdx.x + i * T, m = min(it / IPR, M - 1);
      if constexpr (EPI == DG_RESADD) e_res[i] = *reinterpret_cast<const u16x4*>(a.res + (long)m * a.ldr + min(col0 + it % IPR * 4, N - 4));
      else { e_slot[i] = a.slots[m]; e_pos[i] = a.pos[m]; }
    }
  }

  f32x4 e_bg[EPI == DG_GLU ? NI : 1], e_bu[EPI == DG_GLU ? NI : 1];
  if constexpr (EPI == DG_GLU) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int q = (threadIdx.x + i * T) % IPR, c = min(8 * (tile * NT + q / 2) + 4 * (q & 1), N / 2 - 4);
      e_bg[i] = a.bias ? *reinterpret_cast<const f32x4*>(a.bias + c) : f32x4{0.f, 0.f, 0.f, 0.f};
      e_bu[i] = a.bias ? *reinterpret_cast<const f32x4*>(a.bias + N / 2 + c) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }

  f32x4 acc[MT][NT], sq[SQ ? MT : 1];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (SQ) sq[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int nt16 = (N + 15) >> 4;
  __amdgpu_buffer_rsrc_t wt[NT];      // a tile's weights up to the wave's last k: reads behind it are zeros that cost no traffic
#pragma unroll
  for (int n = 0; n < NT; ++n) wt[n] = make_rsrc(a.W + (long)min(tile * NT + n, nt16 - 1) * 16 * K, (unsigned)wk1 * 32);
  // X: fragments (row r16, 8 k of group g), or rows (XL): 4 U lanes a row
  constexpr int LR = 4 * U, RPI = 64 / LR;
  const int xr = XL ? lane / LR : r16, xc = XL ? lane % LR : g;
  // (rows past M read as zeros: out of the buffer's range)
  const __amdgpu_buffer_rsrc_t xb = make_rsrc(a.X, (unsigned)(((long)(M - 1) * a.ldx + K) * 2));
  const unsigned x0 = (unsigned)(xr * (int)a.ldx + 8 * xc) * 2;
  unsigned char* mine = dg_smem + wave * C::REG;

  // A stage's rows first: they go through LDS while its weights are on their way.  No load stands behind a condition (past the wave's
  // k they are out of the buffers' ranges): where ways with and without a load meet, the compiler waits for all that are in flight, and
  // with `if (there is a next stage) load` in the loop it had one stage's latency for every two.  us in a captured graph, weights from HBM, 48
  // rows: 11264 x 2048 SwiGLU 13.0 -> 11.8, 2560 x 2048 QKV 8.4 -> 7.6, 2048 x 2048 6.8 -> 6.6, 2048 x 5632 10.2 -> 10.1; 16 rows 10.3 -> 9.8, 6.0 -> 5.7,
  // 8.9 -> 8.6 (the last).  Three stages of two steps: 12.3, 7.7, 6.9, 10.0.
  struct Stage { bf16x8 w[U][NT]; uint4 x[U * MT]; };
  auto load = [&](Stage& st, int k0, auto cnt) {      // the first cnt steps of a stage
    keep_order();
    const unsigned wo = (unsigned)(k0 * 32 + lane * 16), xo = k0 < wk1 ? x0 + (unsigned)k0 * 2 : 0x40000000u;
    if constexpr (XL) {
      // (a short stage reads on into other k: never multiplied)
#pragma unroll
      for (int i = 0; i < U * MT; ++i) st.x[i] = ldb16(xb, xo + (unsigned)(RPI * i * (int)a.ldx) * 2);
    }
    keep_order();
#pragma unroll
    for (int u = 0; u < cnt.value; ++u) {
#pragma unroll
      for (int n = 0; n < NT; ++n) st.w[u][n] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wt[n], wo + u * 1024, 0, 2));
      if constexpr (!XL) st.x[u] = ldb16(xb, xo + u * 64);
    }
    keep_order();
  };
  auto compute = [&](const Stage& st, int cnt, auto most) {
    if constexpr (XL) {
#pragma unroll
      for (int i = 0; i < U * MT; ++i) *reinterpret_cast<uint4*>(mine + (RPI * i + xr) * PX + xc * 16) = st.x[i];
    }
#pragma unroll
    for (int u = 0; u < most.value; ++u)
      if (u < cnt) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          bf16x8 xf;
          if constexpr (XL) xf = *reinterpret_cast<const bf16x8*>(mine + (16 * m + r16) * PX + (4 * u + g) * 16);
          else xf = __builtin_bit_cast(bf16x8, st.x[u]);
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, st.w[u][n], acc[m][n], 0, 0, 0);
          if constexpr (SQ) sq[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, xf, sq[m], 0, 0, 0);
        }
      }
  };
  float4 e_co[EPI == DG_QKV ? NI : 1], e_si[EPI == DG_QKV ? NI : 1];
  auto angles = [&] {      // behind the first weights
    if constexpr (EPI == DG_QKV) {
      const int hd = a.d / 2, qk = (a.nq + a.nkv) * a.d;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int it = (threadIdx.x + i * T) % IPR, t16 = tile * NT + it / 2, cb = (t16 >> 1) * 32;
        if (cb < qk) {
          const int d1 = 16 * ((cb % a.d) >> 5) + 8 * (t16 & 1) + 4 * (it & 1);
          const float* cs = a.cos_sin + (long)e_pos[i] * a.d + d1;
          e_co[i] = *reinterpret_cast<const float4*>(cs);
          e_si[i] = *reinterpret_cast<const float4*>(cs + hd);
        }
      }
    }
  };
  const int steps = (wk1 - wk0) / 32;
  constexpr std::integral_constant<int, U> whole{};
  constexpr std::integral_constant<int, U / 2> half{};
  if (steps <= 0) {      // a wave without k: a group past the last split
    angles();
  } else {
    Stage A, B;
    if constexpr (HALVES == 1) load(A, wk0, half);
    else load(A, wk0, whole);
    if constexpr (HALVES == 3) load(B, wk0 + 32 * U, half);
    if constexpr (HALVES == 0) load(B, wk0 + 32 * U, whole);
    angles();
    if constexpr (HALVES == 0) {
      int i = 0;
      for (; i + 2 * U < steps; i += 2 * U) {
        compute(A, U, whole);
        load(A, wk0 + (i + 2 * U) * 32, whole);
        compute(B, U, whole);
        load(B, wk0 + (i + 3 * U) * 32, whole);
      }
      if (steps > i) compute(A, steps - i, whole);
      if (steps > i + U) compute(B, steps - i - U, whole);
    } else {
      if constexpr (HALVES == 1) compute(A, steps, half);
      else compute(A, steps, whole);
      if constexpr (HALVES == 3) compute(B, steps - U, half);
    }
  }

  // ---- the waves' partial tiles meet in LDS (each wave's own piece: its staged rows are read).  acc[m][n][r] = C[16m + 4g + r][16n + r16]
  float* pt = reinterpret_cast<float*>(mine);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) pt[(16 * m + 4 * g + r) * LD + 16 * n + r16] = acc[m][n][r];
    if constexpr (SQ) {
      const float dg = r16 & 2 ? (r16 & 1 ? sq[m][3] : sq[m][2]) : (r16 & 1 ? sq[m][1] : sq[m][0]);
      if ((r16 >> 2) == g) s_tail[wave * MR + 16 * m + r16] = dg;
    }
  }
  __syncthreads();
  auto group_part = [&](int gr, int row, int c) {
    const unsigned char* b = dg_smem + gr * 4 * C::REG + (row * LD + c) * 4;
    auto at = [&](int w) { return *reinterpret_cast<const f32x4*>(b + w * C::REG); };
    return (at(0) + at(2)) + (at(1) + at(3));
  };
  auto group_sum = [&](int row, int c) {
    f32x4 v = group_part(0, row, c);
    if constexpr (VS > 1) {
      v += 0.f;      // as a sum of slabs begins
#pragma unroll
      for (int gr = 1; gr < VS; ++gr) v += group_part(gr, row, c);
    }
    return v;
  };
  auto row_sum = [&](int w0, int n, int row) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < n; ++w) s += s_tail[(w0 + w) * MR + row];
    return s;
  };
  f32x4 x1[NI], x2[PAIR ? NI : 1];
  float rs[SQ ? NI : 1];
  if (gridDim.y > 1) {
    // write-through slabs, one a split (results, then the rows' sums), ticket; the last arriver adds them in split order
    constexpr int slab = MR * NC + (SQ ? MR : 0);
    const int S = gridDim.y * VS;
    const __amdgpu_buffer_rsrc_t pr = make_rsrc(a.part, (unsigned)min((long)gridDim.x * S * slab * 4, 0x7fffffffL));
    auto slab_at = [&](int sp) { return (unsigned)(((long)sp * gridDim.x + tile) * slab * 4); };
#pragma unroll
    for (int gr = 0; gr < VS; ++gr) {
      const unsigned my = slab_at(blockIdx.y * VS + gr);
      for (int e = threadIdx.x * 4; e < min(M, MR) * NC; e += T * 4) {
        const f32x4 v = group_part(gr, e / NC, e % NC);
        st_wt16(pr, my + e * 4, make_float4(v[0], v[1], v[2], v[3]));
      }
      if constexpr (SQ)
        if (threadIdx.x < MR / 4) {
          const int m = threadIdx.x * 4;
          st_wt16(pr, my + (MR * NC + m) * 4, make_float4(row_sum(4 * gr, 4, m), row_sum(4 * gr, 4, m + 1), row_sum(4 * gr, 4, m + 2), row_sum(4 * gr, 4, m + 3)));
        }
    }
    if (!ticket_last(&a.counters[tile], gridDim.y, s_last)) return;
    auto all_slabs = [&](int e) {
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
      for (int sp = 0; sp < S; ++sp) {
        const float4 q = ld_wt16(pr, slab_at(sp) + e * 4);
        v += f32x4{q.x, q.y, q.z, q.w};
      }
      return v;
    };
    if constexpr (SQ) {
      if (threadIdx.x < MR / 4) *reinterpret_cast<f32x4*>(s_tail + threadIdx.x * 4) = all_slabs(MR * NC + threadIdx.x * 4);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int it = threadIdx.x + i * T, row = it / IPR, q = it % IPR;
      if (row >= M) continue;
      if constexpr (PAIR) {
        x1[i] = all_slabs(row * NC + q / 2 * 16 + 4 * (q & 1));
        x2[i] = all_slabs(row * NC + q / 2 * 16 + 8 + 4 * (q & 1));
      } else x1[i] = all_slabs(row * NC + 4 * q);
    }
    if constexpr (SQ) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NI; ++i) rs[i] = s_tail[min((int)(threadIdx.x + i * T) / IPR, MR - 1)];
    }
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int it = threadIdx.x + i * T, row = it / IPR, q = it % IPR;
      if (row >= M) continue;
      if constexpr (PAIR) {
        x1[i] = group_sum(row, q / 2 * 16 + 4 * (q & 1));
        x2[i] = group_sum(row, q / 2 * 16 + 8 + 4 * (q & 1));
        if constexpr (SQ) rs[i] = row_sum(0, WV, row);
      } else x1[i] = group_sum(row, 4 * q);
    }
    if constexpr (EPI == DG_RESADD) __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int it = threadIdx.x + i * T, m = it / IPR, q = it % IPR;
    if (m >= M) continue;
    u16x4 o;
    if constexpr (EPI == DG_PLAIN || EPI == DG_GELU) {
      const int c = col0 + 4 * q;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o.v[j] = f2bf(x1[i][j]);
        if constexpr (EPI == DG_GELU) {
          const float v = bf2f(o.v[j]);
          o.v[j] = f2bf(gelu_bf(v));
        }
      }
      u16* y = a.Y + (long)m * a.ldy + c;
      if (c + 4 <= N && (a.ldy & 3) == 0) *reinterpret_cast<u16x4*>(y) = o;
      else
        for (int j = 0; j < 4; ++j)
          if (c + j < N) y[j] = o.v[j];
    } else if constexpr (EPI == DG_RESADD) {
      // r = bf16(bf16(acc) + r) (res_add_ssq numerics)
      const int c = col0 + 4 * q;
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = bf2f(f2bf(bf2f(f2bf(x1[i][j])) + bf2f(e_res[i].v[j])));
        o.v[j] = f2bf(v);
        ss += v * v;
      }
      if (c < N) *reinterpret_cast<u16x4*>(a.res + (long)m * a.ldr + c) = o;
      s_tail[m * (NC / 4) + q] = c < N ? ss : 0.f;
    } else if constexpr (EPI == DG_GLU) {
      // the product's rounding, then glu_act's steps (seqmix.hip) on it
      const int c = 8 * (tile * NT + q / 2) + 4 * (q & 1);
      if (2 * c >= N) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float g = bf2f(f2bf(x1[i][j])) + e_bg[i][j], u = bf2f(f2bf(x2[i][j])) + e_bu[i][j], al = 1.f;
        if (a.mode == 1) {
          g = fminf(g, a.limit);
          u = fminf(fmaxf(u, -a.limit), a.limit) + 1.f;
          al = a.alpha;
        } else if (a.mode == 2) {
          al = 1.5957691216057308f * (1.f + 0.044715f * g * g);
        }
        o.v[j] = f2bf(g * __builtin_amdgcn_rcpf(1.f + __expf(-al * g)) * u);
      }
      *reinterpret_cast<u16x4*>(a.Y + (long)m * a.ldy + c) = o;
    } else {
      const float ri = rsqrtf(rs[i] * a.scale + a.eps);
      const int t16 = tile * NT + q / 2, h8 = 8 * (t16 & 1) + 4 * (q & 1), cb = (t16 >> 1) * 32;
      if (cb >= N) continue;
      if constexpr (EPI == DG_SWIGLU) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float gv = bf2f(f2bf(x1[i][j] * ri)), uv = bf2f(f2bf(x2[i][j] * ri));
          o.v[j] = f2bf(gv / (1.f + __expf(-gv)) * uv);
        }
        *reinterpret_cast<u16x4*>(a.Y + (long)m * a.ldy + cb / 2 + h8) = o;
      } else {
        const int d = a.d, hd = d / 2, qcols = a.nq * d, kcols = a.nkv * d, slot = e_slot[i];
        const long blk = slot >> 4, off = slot & 15;
        float b1[4], b2[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) { b1[j] = bf2f(f2bf(x1[i][j] * ri)); b2[j] = bf2f(f2bf(x2[i][j] * ri)); }
        if (cb < qcols + kcols) {
          const bool isq = cb < qcols;
          const int cc = isq ? cb : cb - qcols, head = cc / d, d1 = 16 * ((cc % d) >> 5) + h8;
          const float co[4] = {e_co[i].x, e_co[i].y, e_co[i].z, e_co[i].w}, si[4] = {e_si[i].x, e_si[i].y, e_si[i].z, e_si[i].w};
          u16* dst = isq ? a.q_out + ((long)m * a.nq + head) * d
                         : (slot >= 0 ? a.kc + ((blk * a.nkv + head) * 16 + off) * d : nullptr);
          if (dst) {
            u16x4 o2;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              o.v[j] = f2bf(b1[j] * co[j] - b2[j] * si[j]);
              o2.v[j] = f2bf(b2[j] * co[j] + b1[j] * si[j]);
            }
            *reinterpret_cast<u16x4*>(dst + d1) = o;
            *reinterpret_cast<u16x4*>(dst + hd + d1) = o2;
          }
        } else {
          const int cc = cb - qcols - kcols + h8;
          u16x4 o2;
#pragma unroll
          for (int j = 0; j < 4; ++j) { o.v[j] = f2bf(b1[j]); o2.v[j] = f2bf(b2[j]); }
          if (a.v_rows) {
            *reinterpret_cast<u16x4*>(a.v_rows + (long)m * a.v_ld + cc) = o;
            *reinterpret_cast<u16x4*>(a.v_rows + (long)m * a.v_ld + cc + 16) = o2;
          } else if (slot >= 0) {
            u16* vo = a.vc + ((blk * a.nkv + cc / d) * d + cc % d) * 16 + off;
#pragma unroll
            for (int j = 0; j < 4; ++j) { vo[j * 16] = o.v[j]; vo[(16 + j) * 16] = o2.v[j]; }
          }
        }
      }
    }
  }
  if constexpr (EPI == DG_RESADD) {
    __syncthreads();
    if (threadIdx.x < min(M, MR)) {
      float ss = 0.f;
      for (int c = 0; c < NC / 4; ++c) ss += s_tail[threadIdx.x * (NC / 4) + c];      // fixed order
      a.ssq_out[(long)tile * a.ssq_ld + threadIdx.x] = ss;
    }
  }
}

template <int MT, int NT, int VS, int EPI, int HALVES>
int raise_lds() {
  return (int)hipFuncSetAttribute((const void*)dgemm_kernel<MT, NT, VS, EPI, HALVES>, hipFuncAttributeMaxDynamicSharedMemorySize, Dg<MT, NT, VS, EPI>::LDS);
}

template <int MT, int NT, int VS, int EPI>
int launch(const DgArgs& a, int gy, hipStream_t st) {
  using C = Dg<MT, NT, VS, EPI>;
  static_assert(C::LDS <= 160 * 1024, "LDS of a workgroup");
  // raised once, for every length of K: no attribute call inside a later stream capture
  static const int rc = C::LDS <= 64 * 1024 ? 0 : raise_lds<MT, NT, VS, EPI, 0>() | raise_lds<MT, NT, VS, EPI, 1>() |
                                                      raise_lds<MT, NT, VS, EPI, 2>() | raise_lds<MT, NT, VS, EPI, 3>();
  if (rc) return rc;
  const dim3 grid((a.N + C::NC - 1) / C::NC, gy);
  constexpr int H = C::U / 2;
  switch ((((a.kchunk + 3) / 4 + 31) / 32 + H - 1) / H) {      // half stages of the longest wave
    case 1: hipLaunchKernelGGL((dgemm_kernel<MT, NT, VS, EPI, 1>), grid, dim3(C::T), C::LDS, st, a); break;
    case 2: hipLaunchKernelGGL((dgemm_kernel<MT, NT, VS, EPI, 2>), grid, dim3(C::T), C::LDS, st, a); break;
    case 3: hipLaunchKernelGGL((dgemm_kernel<MT, NT, VS, EPI, 3>), grid, dim3(C::T), C::LDS, st, a); break;
    default: hipLaunchKernelGGL((dgemm_kernel<MT, NT, VS, EPI, 0>), grid, dim3(C::T), C::LDS, st, a);
  }
  return (int)hipGetLastError();
}

template <int MT, int EPI>
int by_shape(const DgArgs& a, int nt, int vs, int gy, hipStream_t st) {
  if (vs == 1) {
    if (nt == 1) return launch<MT, 1, 1, EPI>(a, gy, st);
    if (nt == 2) return launch<MT, 2, 1, EPI>(a, gy, st);
    if (nt == 3) return launch<MT, 3, 1, EPI>(a, gy, st);
  } else if (vs == 2) {
    if (nt == 1) return launch<MT, 1, 2, EPI>(a, gy, st);
    if (nt == 2) return launch<MT, 2, 2, EPI>(a, gy, st);
    if (nt == 3) return launch<MT, 3, 2, EPI>(a, gy, st);
  } else if (vs == 4) {
    if constexpr (MT <= 2 && (EPI == DG_PLAIN || EPI >= DG_GLU))
      if (nt == 1) return launch<MT, 1, 4, EPI>(a, gy, st);
  }
  return -10;
}

template <int EPI>
int by_rows(const DgArgs& a, int nt, int vs, int gy, hipStream_t st) {
  if (a.M <= 16) return by_shape<1, EPI>(a, nt, vs, gy, st);
  if (a.M <= 32) return by_shape<2, EPI>(a, nt, vs, gy, st);
  if (a.M <= 48) return by_shape<3, EPI>(a, nt, vs, gy, st);
  return by_shape<4, EPI>(a, nt, vs, gy, st);
}
}  // namespace

// W: ops.gemm.frag_weight's [ceil(N / 16)][K / 32][64][8], paired for QKV / SWIGLU.  nt 16-column tiles a workgroup, splits of K: vs of
// them in a workgroup.  With gy = ceil(splits / vs) > 1 workgroups a tile, part holds gy vs slabs of 16 ceil(M / 16) (16 nt + 1) floats per
// tile, counters one zeroed int per tile.  RESADD writes ceil(N / (16 nt)) row-sum slots.
extern "C" int dllm_dgemm(const void* X, long ldx, const void* W, void* Y, long ldy, int M, int N, int K, int nt, int vs, int splits,
                          int epi, float* part, int* counters, void* res, long ldr, float* ssq_out, long ssq_ld, float scale, float eps,
                          const int* pos, const float* cos_sin, const int* slots, void* q_out, void* kc, void* vc, void* v_rows,
                          long v_ld, int nq, int nkv, int d, const float* bias, int mode, float limit, float alpha, hipStream_t stream) {
  if (M < 1 || M > 64 || ldx < K || ldx > (1 << 24) || N < 1 || K < 32 || K % 32 || splits < 1 || nt < 1 || vs < 1) return -1;
  int kchunk = (K + splits - 1) / splits;
  kchunk = (kchunk + 31) & ~31;
  const int S = (K + kchunk - 1) / kchunk, gy = (S + vs - 1) / vs;
  if (gy > 1 && (!part || !counters)) return -2;
  const DgArgs a{(const u16*)X, ldx, (const u16*)W, (u16*)Y, ldy, M, N, K, kchunk, S, part, counters, (u16*)res, ldr, ssq_out, ssq_ld,
                 scale, eps, pos, cos_sin, slots, (u16*)q_out, (u16*)kc, (u16*)vc, (u16*)v_rows, v_ld, nq, nkv, d,
                 bias, mode, limit, alpha};
  switch (epi) {
    case DG_PLAIN: return Y ? by_rows<DG_PLAIN>(a, nt, vs, gy, stream) : -3;
    case DG_RESADD: return res && ssq_out && N % 4 == 0 && ldr % 4 == 0 ? by_rows<DG_RESADD>(a, nt, vs, gy, stream) : -4;
    case DG_QKV:
      if (d < 32 || d % 32 || N != (nq + 2 * nkv) * d || !q_out || !kc || !vc || !pos || !cos_sin || !slots || (v_rows && v_ld % 4)) return -5;
      return by_rows<DG_QKV>(a, nt, vs, gy, stream);
    case DG_SWIGLU: return Y && N % 32 == 0 && ldy % 4 == 0 ? by_rows<DG_SWIGLU>(a, nt, vs, gy, stream) : -6;
    case DG_GLU: return Y && N % 16 == 0 && ldy % 4 == 0 && mode >= 0 && mode <= 2 ? by_rows<DG_GLU>(a, nt, vs, gy, stream) : -8;
    case DG_GELU: return Y ? by_rows<DG_GELU>(a, nt, vs, gy, stream) : -3;
    default: return -7;
  }
}
