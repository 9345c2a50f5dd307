// Prompt-size products on 256 x 256 tiles of four waves:  Y = epilogue(X[M, K] . W[N, K]^T), bf16 in, f32 accumulate.
//
// What bounded the 256 x 256 tile of eight waves (tgemm.hip) is LDS: a wave of 128 x 64 reads (128 + 64) rows for 128 x 64 outputs, so a
// 32-deep step of the workgroup is 96 KB out of LDS and 32 KB into it, as many cycles at 128 B a clock as its products take, and the
// two waves of a SIMD read at the same time and multiply at the same time.  Four waves of 128 x 128, one a SIMD, read a third less, and each
// keeps its matrix core busy by itself: the fragments of the next half step are read, and the tile after the next is requested,
// between the products of this one.
//   * Ring of two 64-deep stages; a half step is 64 products (16 x 16 x 32) over one of two register sets of fragments.  First half:
//     multiply k 0..31, read k 32..63; once every wave has them (barrier) the stage is free and its refill begins.  Second half: multiply
//     k 32..63, read k 0..31 of the next stage (landed: counted vmcnt ahead of a second barrier), the rest of the refill.
//   * 256 accumulators a lane are all of its AGPRs.  The compiler then copies accumulators round (three moves a product), so
//     the product is one inline instruction that adds in place, and the order of products, reads and refills is the one written here.
//   * W is the products' first operand: a lane holds four neighbouring outputs of one row, two fragments of a row become 16 bytes
//     by two row swaps, and results leave from registers in 64-byte pieces of a row.  (Staged through LDS in 2-byte stores and copied out, a
//     tile of 128-deep K took 15 us, of which its products are two.)
// us, here / eight waves (the vendor's plain product): 7936 x 11264 x 2048 with SwiGLU 310 / 371 (319); 8192 x 2048 x 5632 134 / 158 (121), 1.41
// PFLOP/s; 16128 x 2048 x 1024 62 / 70 (56).  Experts of a prompt (8048 tokens, 8 of 1024 x 1024, top 2) 173 / 205.
#include <type_traits>

#include "common.h"
#include "tgemm_shared.h"

typedef __attribute__((address_space(3))) void lds_void;

namespace {
using namespace dllm;

constexpr int KD = 64, ROW = 2 * KD;      // k depth of a stage, bytes of a staged row
// (bytes 16 c of row r lie at chunk c ^ swizzle(r): the 16 rows of a fragment read meet no bank twice; tgemm.hip)
__device__ __forceinline__ int swizzle(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ float silu(float x) { return x / (1.f + __expf(-x)); }
__device__ __forceinline__ float bfr(float x) { return bf2f(f2bf(x)); }

// Two fragments of a row (a lane holds columns 4 g .. 4 g + 3 of each): 16 bytes, columns 16 (g & 1) + 8 (g >> 1) .. + 7 of the 32
__device__ __forceinline__ uint4 join(const float* a, const float* b) {
  const auto x = __builtin_amdgcn_permlane16_swap(f2bf2(a[0], a[1]), f2bf2(b[0], b[1]), false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(f2bf2(a[2], a[3]), f2bf2(b[2], b[3]), false, false);
  return make_uint4(x[0], y[0], x[1], y[1]);
}

template <int EPI>
__global__ void __launch_bounds__(256) wide_gemm_kernel(GemmArgs a) {
  constexpr int F = 8, BM = 256, BN = 256, NT = 256, G = 2 * F;      // fragments a side of a wave tile; ring loads a wave and stage
  constexpr int A_BYTES = BM * ROW, STAGE = (BM + BN) * ROW, OLD = BN + 8;
  constexpr int RING = EPI == EPI_QKV ? BM * OLD * 2 : 2 * STAGE;
  static_assert(RING >= 2 * STAGE, "the staged rows of the QKV epilogue lie over the ring");
  __shared__ __attribute__((aligned(16))) unsigned char smem[RING + 4 * BM * 4];
  float* s_rinv = reinterpret_cast<float*>(smem + RING);      // [BM] row scales; RESADD: [2][BM] row sums
  int* s_slot = reinterpret_cast<int*>(s_rinv + BM);
  int *s_pos = s_slot + BM, *s_run = s_slot + 2 * BM;

  // XCD-aware remap and grouped raster, as tgemm_kernel
  const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN, nwg = mt * nt, q8 = nwg >> 3, r8 = nwg & 7, xcd = blockIdx.x & 7;
  const int wg = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (blockIdx.x >> 3);
  int m_t = wg % mt, n_t = wg / mt;
  if (a.raster > 1 && mt > a.raster) {
    const int gsz = a.raster * nt, first = (wg / gsz) * a.raster, gm = min(mt - first, a.raster), in = wg % gsz;
    m_t = first + in % gm;
    n_t = in / gm;
  }
  int m0 = m_t * BM, M = a.M;
  const int n0 = n_t * BN, N = a.N, K = a.K, nk = K / KD;
  const u16* Wb = a.W;
  if (a.g_tiles != nullptr) {      // grouped (experts): row tile from the device list (block-uniform exit)
    if (m_t >= a.g_tiles[3 * a.g_max]) return;
    m0 = a.g_tiles[a.g_max + m_t];
    M = m0 + a.g_tiles[2 * a.g_max + m_t];
    Wb = a.W + (long)a.g_tiles[m_t] * a.g_wstride;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
  const int g = lane >> 4, r16 = lane & 15;

  // what the epilogue needs of the tile's rows (a thread a row), requested ahead of the ring: back at its first wait
  constexpr bool SCALED = EPI == EPI_QKV || EPI == EPI_SWIGLU || EPI == EPI_PLAIN;
  const bool has_rs = SCALED && a.ssq_in != nullptr;
  const int my = min(m0 + (int)threadIdx.x, M - 1);
  float ssv[8];
  if (has_rs) {
#pragma unroll
    for (int u = 0; u < 8; ++u) ssv[u] = a.ssq_in[(long)min(u, a.ssq_in_n - 1) * a.ssq_in_ld + my] * (u < a.ssq_in_n ? 1.f : 0.f);
  }
  int q_pos = 0, q_slot = 0;
  if constexpr (EPI == EPI_QKV) { q_pos = a.pos[my]; q_slot = a.slots[my]; }

  // ring: a wave's load is 1 KB, eight staged rows; lane -> row lane / 8, LDS chunk lane % 8 <- source chunk ^ swizzle(row)
  const int srow = lane >> 3, spos = lane & 7;
  const bool wp = a.w_panel != 0;      // K-panel-major weights
  const u16 *a_src[F], *b_src[F];
#pragma unroll
  for (int j = 0; j < F; ++j) {
    const int r = 8 * (wave * F + j) + srow, c = 8 * (spos ^ swizzle(r)), row = min(m0 + r, M - 1);
    a_src[j] = a.A + (a.g_perm != nullptr ? (long)(a.g_perm[row] / a.g_k) : (long)row) * a.lda + c;
    const long n = min(n0 + r, N - 1);
    b_src[j] = Wb + (wp ? n * KD : n * K) + c;
  }
  auto request = [&](int t, int q) {      // load q of the wave's G for stage t
    unsigned char* base = smem + (t & 1) * STAGE;
    if (q < F) __builtin_amdgcn_global_load_lds((const void*)(a_src[q] + t * KD), (lds_void*)(base + (wave * F + q) * 1024), 16, 0, 0);
    else __builtin_amdgcn_global_load_lds((const void*)(b_src[q - F] + (wp ? (long)t * KD * N : (long)t * KD)),
                                          (lds_void*)(base + A_BYTES + (wave * F + q - F) * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int q = 0; q < G; ++q) request(0, q);
  if (nk > 1) {
#pragma unroll
    for (int q = 0; q < G; ++q) request(1, q);
  }
  if (has_rs) {
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) s += ssv[u];
    for (int b = 8; b < a.ssq_in_n; b += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) s += a.ssq_in[(long)min(b + u, a.ssq_in_n - 1) * a.ssq_in_ld + my] * (b + u < a.ssq_in_n ? 1.f : 0.f);
    }
    s_rinv[threadIdx.x] = rsqrtf(s * a.norm_scale + a.eps);
  }
  if constexpr (EPI == EPI_QKV) { s_slot[threadIdx.x] = q_slot; s_pos[threadIdx.x] = q_pos; }

  f32x4 acc[F][F];      // acc[i][j][e] = C[16 i + r16][16 j + 4 g + e] of the wave tile
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));      // written here, well ahead of an inline product that reads it
    }

  bf16x8 x0[F], w0[F], x1[F], w1[F];      // fragments of k 0..31 and 32..63 of a stage
  const int ra = wm * 16 * F + r16, rb = wn * 16 * F + r16;
  const int ca = (g ^ swizzle(ra)) << 4, cb = (g ^ swizzle(rb)) << 4;
  // W and X of half h of stage t, fragment q of 2 F (the products take a row of fragments of W first)
  auto read = [&](bf16x8* x, bf16x8* w, int t, int h, int q) {
    const unsigned char* base = smem + (t & 1) * STAGE;
    if (q < F) w[q] = *reinterpret_cast<const bf16x8*>(base + A_BYTES + (rb + 16 * q) * ROW + (cb ^ (64 * h)));
    else x[q - F] = *reinterpret_cast<const bf16x8*>(base + (ra + 16 * (q - F)) * ROW + (ca ^ (64 * h)));
  };
  auto mul4 = [&](const bf16x8* x, const bf16x8* w, int q) {
#pragma unroll
    for (int u = 4 * q; u < 4 * q + 4; ++u)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[u / F][u % F]) : "v"(w[u % F]), "v"(x[u / F]));
  };
  constexpr int GROUPS = F * F / 4, EARLY = 6;      // groups of four products a half step; loads of a refill in its first half
  auto step = [&](int t, auto refill, auto next) {
#pragma unroll
    for (int q = 0; q < GROUPS; ++q) {
      mul4(x0, w0, q);
      if (q < F) { read(x1, w1, t, 1, 2 * q); read(x1, w1, t, 1, 2 * q + 1); }
      if (q == GROUPS - EARLY - 1) {
        __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0): this wave's reads of the stage
        __builtin_amdgcn_s_barrier();
      }
      if constexpr (refill.value)
        if (q >= GROUPS - EARLY) request(t + 2, q - (GROUPS - EARLY));
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70 | (refill.value ? EARLY : 0));      // vmcnt: the next stage's loads, issued a step ago
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < GROUPS; ++q) {
      mul4(x1, w1, q);
      if constexpr (refill.value)
        if (q < G - EARLY) request(t + 2, q + EARLY);
      if constexpr (next.value)
        if (q < F) { read(x0, w0, t + 1, 0, 2 * q); read(x0, w0, t + 1, 0, 2 * q + 1); }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  static_assert(G == GROUPS && G - EARLY <= GROUPS && F < GROUPS - EARLY, "a read and a load beside every four products");
  if (nk > 1) __builtin_amdgcn_s_waitcnt(0x0070 | (G & 15) | (G >> 4 << 14));      // vmcnt(G) lgkmcnt(0): stage 0 has landed
  else __builtin_amdgcn_s_waitcnt(0x0070);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < G; ++q) read(x0, w0, 0, 0, q);
  for (int t = 0; t + 2 < nk; ++t) step(t, std::true_type{}, std::true_type{});
  if (nk > 1) step(nk - 2, std::false_type{}, std::true_type{});
  step(nk - 1, std::false_type{}, std::false_type{});
  // the compiler does not know when an inline product's result can be read: none is read before this point
  asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) asm volatile("" : "+a"(acc[i][j]));

  // ---- epilogue, from registers: row rl + 16 i, columns by fragment pairs
  const int rl = wm * 16 * F + r16, cw = wn * 16 * F;
  if constexpr (EPI == EPI_F32) {
    float* yf = reinterpret_cast<float*>(a.Y);
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j) {
        const int m = m0 + rl + 16 * i, n = n0 + cw + 16 * j + 4 * g;
        if (m < M && n < N) *reinterpret_cast<f32x4*>(yf + (long)m * a.ldy + n) = acc[i][j];
      }
  } else if constexpr (EPI == EPI_QKV) {
    u16* so = reinterpret_cast<u16*>(smem);      // (every read of the ring is behind the last barrier)
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const float ri = has_rs ? s_rinv[rl + 16 * i] : 1.f;
#pragma unroll
      for (int j = 0; j < F; ++j)
        *reinterpret_cast<uint2*>(so + (rl + 16 * i) * OLD + cw + 16 * j + 4 * g) =
            make_uint2(f2bf2(acc[i][j][0] * ri, acc[i][j][1] * ri), f2bf2(acc[i][j][2] * ri, acc[i][j][3] * ri));
    }
    __syncthreads();
    qkv_copy_out<BM, BN, OLD, NT>(a, so, s_slot, s_pos, s_run, M, m0, n0);
  } else {
    const int c8 = 16 * (g & 1) + 8 * (g >> 1);      // where `join` leaves a lane's eight columns
    constexpr int NV = EPI == EPI_SWIGLU ? F / 4 : F / 2;      // 16-byte vectors a row
    const int nc = EPI == EPI_SWIGLU ? (n0 + cw) / 2 : n0 + cw, nlim = EPI == EPI_SWIGLU ? N / 2 : N;
    uint4 res[EPI == EPI_RESADD ? F : 1][NV];
    if constexpr (EPI == EPI_RESADD) {
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const int m = min(m0 + rl + 16 * i, M - 1), n = min(nc + 32 * v + c8, nlim - 8);
          res[i][v] = ld16(a.Y + (long)m * a.ldy + n);
        }
    }
    float bias[EPI == EPI_PLAIN || EPI == EPI_GELU || EPI == EPI_RESADD ? F : 1][4];
    const bool biased = (EPI == EPI_PLAIN || EPI == EPI_GELU || EPI == EPI_RESADD) && a.bias != nullptr;
    if constexpr (EPI == EPI_PLAIN || EPI == EPI_GELU || EPI == EPI_RESADD) {
#pragma unroll
      for (int j = 0; j < F; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) bias[j][e] = biased ? bf2f(a.bias[min(n0 + cw + 16 * j + 4 * g + e, N - 1)]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const int m = m0 + rl + 16 * i;
      const float ri = has_rs ? s_rinv[rl + 16 * i] : 1.f;
      float ss = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        float p[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (EPI == EPI_SWIGLU) {
              const float gv = bfr(acc[i][4 * v + 2 * h][e] * ri), uv = bfr(acc[i][4 * v + 2 * h + 1][e] * ri);
              p[h][e] = silu(gv) * uv;
            } else {
              float x = acc[i][2 * v + h][e] * ri;
              if constexpr (EPI != EPI_RELU2) x += bias[2 * v + h][e];
              if constexpr (EPI == EPI_GELU) x = gelu_bf(bfr(x));      // GELU of the bf16 linear output
              if constexpr (EPI == EPI_RELU2) x = fmaxf(x, 0.f) * fmaxf(x, 0.f);
              p[h][e] = x;
            }
          }
        uint4 o = join(p[0], p[1]);
        const int n = nc + 32 * v + c8;
        const bool in = m < M && n < nlim;
        if constexpr (EPI == EPI_RESADD) {
          float x[8], r[8];
          unpack8(o, x);
          unpack8(res[i][v], r);
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            r[k] = bfr(x[k] + r[k]);
            ss += in ? r[k] * r[k] : 0.f;
          }
          o = pack8(r);
        }
        if (in) st16(a.Y + (long)m * a.ldy + n, o);
      }
      if constexpr (EPI == EPI_RESADD) {
        ss = lane_add(ss, 16);
        ss = lane_add(ss, 32);
        if (g == 0) s_rinv[wn * BM + rl + 16 * i] = ss;      // (the row's half of the tile)
      }
    }
    if constexpr (EPI == EPI_RESADD) {
      __syncthreads();
      const int m = m0 + threadIdx.x;
      if (a.ssq_out != nullptr && m < M) a.ssq_out[(long)n_t * a.ssq_out_ld + m] = s_rinv[threadIdx.x] + s_rinv[BM + threadIdx.x];
    }
  }
}

template <int EPI>
int launch(const GemmArgs& a, hipStream_t st) {
  const int grid = ((a.M + 255) / 256) * ((a.N + 255) / 256);
  hipLaunchKernelGGL((wide_gemm_kernel<EPI>), dim3(grid), dim3(256), 0, st, a);
  return (int)hipGetLastError();
}
}  // namespace

// The 256 x 256 tile of four waves: dllm_tgemm's plan (256, 256, 2 stages, 64 deep, 4 waves), checked there; one split, no stream-K.
int dllm::wide_gemm(const GemmArgs& a, int epi, hipStream_t st) {
  if (a.splits != 1 || a.kchunk < a.K || a.K < KD || a.K % KD || a.sk_table != nullptr || a.N % 8) return -29;
  switch (epi) {
    case EPI_PLAIN: return launch<EPI_PLAIN>(a, st);
    case EPI_RESADD: return launch<EPI_RESADD>(a, st);
    case EPI_QKV: return launch<EPI_QKV>(a, st);
    case EPI_SWIGLU: return launch<EPI_SWIGLU>(a, st);
    case EPI_GELU: return launch<EPI_GELU>(a, st);
    case EPI_RELU2: return launch<EPI_RELU2>(a, st);
    case EPI_F32: return launch<EPI_F32>(a, st);
    default: return -6;
  }
}
