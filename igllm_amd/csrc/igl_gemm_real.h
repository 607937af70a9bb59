// igl_gemm_real.h - a real plane (bf16 or binary16 rows) times five lanes
// of fp32 activations and more, gfx950 bf16 MFMA.
//
// C[m][n] = sum_k x[m][k] * w[n][k], the PLANE_REAL arm of back_mat_mat
// (app_core.c:5247-5323 over 4239-4248), for the lane counts where
// gemv_real_kernel's eight lanes a launch would read the plane again and
// again.
//
// Every product is exact, as an fp32 FMA's is.  An fp32 activation is the sum
// of three bf16 terms, each the top sixteen bits of what the terms before it
// left (8 + 8 + 8 significand bits, no rounding, bf16's exponent range is
// fp32's); a bf16 weight is one term and a binary16 weight two (8 + 3 bits).
// A product of two terms is exact in fp32, and v_mfma_f32_16x16x32_bf16 adds
// it into an fp32 accumulator.  An output that comes out infinite or NaN (an
// infinite or NaN value among its operands: a zero term against an infinity), or
// so small that the terms may have cut its activations off (out_of_terms), is
// formed again by plain fp32 FMAs over the row, which is what gemv_real_kernel
// gives.
//
// Rounding.  One accumulator over all of K measured 4.2e-7 off the 64-bit
// product at K = 1536 (N(0,1) activations, 2-norm): the matrix core rounds
// the accumulator about four times an instruction, at its full magnitude.
// The first terms' products are therefore chained over four steps only, from
// zero, and the finished chains added in fp32; the other terms' products, 2^-8
// of it, have an accumulator of their own.  That measures 0.6-1.0e-7 over K
// 256-2048, gemv_real_kernel 0.8-1.2e-7.
//
// What bounds it: below a hundred lanes the plane's stream and the chain of a
// stage (DMA, LDS read, split, products); above, the workgroups' reads of LDS
// and the split between the barriers.  8960 x 1536 bf16, replayed, us, against
// gemv_real_kernel: 5 lanes 18.0 -> 8.6, 16 lanes 32.3 -> 8.8, 64 lanes 112 ->
// 15.1, 500 lanes 848 -> 57 (13.8 GFLOP, three products each: 725 TFLOP/s on
// the matrix cores); binary16 500 lanes 1002 -> 108.
//
// Tiling.  A workgroup of WN x WM x KS waves owns a TN x TM tile of C
// (TN = 16 NB WN weight rows, TM = 16 MB WM lanes).  K advances through LDS
// stages of KS 32-wide steps, written only by the LDS DMA; wave group ks takes
// the ks-th step of a stage, and the KS partial tiles are added in ks order at
// the end.  The waves of a tile lie along the lanes, so no two of them split
// the same activations.
#pragma once

#include "igl_device.h"
#include "igl_launch.h"

namespace igl {

typedef __attribute__((address_space(3))) void real_lds_t;
typedef __attribute__((address_space(1))) const void real_global_t;
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

constexpr int kRealStep = 32;  // k of one wave step: one MFMA

struct GemmRealArgs {
  const float *act;  // 16-byte aligned, act_stride % 4 == 0
  int act_stride;
  const uint16_t *rows;  // [N][K] bf16 or binary16, 16-byte aligned
  float *out;
  int out_stride;
  int M, N, K;  // K % 32 == 0
};

constexpr int real_round(int v, int q) { return (v + q - 1) / q * q; }

template <int WN, int WM, int KS, int NB, int MB, int STAGES>
struct RealForm {
  static constexpr int W = WN * WM * KS;
  static constexpr int TN = 16 * NB * WN;
  static constexpr int TM = 16 * MB * WM;
  static constexpr int A_PAD = real_round(KS * TM * 128, 1024 * W);
  static constexpr int W_PAD = real_round(KS * TN * 64, 1024 * W);
  static constexpr int STAGE = A_PAD + W_PAD;
  static constexpr int RED = (KS - 1) * TN * TM * 4;
  static constexpr int LDS = STAGES * STAGE > RED ? STAGES * STAGE : RED;
  static constexpr int NA = A_PAD / (1024 * W);
  static constexpr int NW = W_PAD / (1024 * W);
  static constexpr int LOADS = NA + NW;
  static_assert(LDS <= 160 * 1024, "LDS");
  static_assert(LOADS * (STAGES - 2) < 64, "vmcnt");
};

// Waits until this wave's loads but the last N are in (vmcnt retires them in
// issue order) and its LDS reads have landed.
template <int N>
__device__ __forceinline__ void real_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt holds six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70);
}

// The high halves of two fp32 values as a pair of bf16, the first one low.
__device__ __forceinline__ uint32_t high_pair(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

__device__ __forceinline__ float high_part(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }

// Eight fp32 values as three bf16 terms each.
__device__ __forceinline__ void split3(const float4_t lo, const float4_t hi, bf8_t (&t)[3]) {
  uint4_t p0, p1, p2;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = i < 2 ? lo[2 * i] : hi[2 * i - 4], b = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
    const float ra = a - high_part(a), rb = b - high_part(b);
    p0[i] = high_pair(a, b);
    p1[i] = high_pair(ra, rb);
    p2[i] = high_pair(ra - high_part(ra), rb - high_part(rb));
  }
  t[0] = __builtin_bit_cast(bf8_t, p0);
  t[1] = __builtin_bit_cast(bf8_t, p1);
  t[2] = __builtin_bit_cast(bf8_t, p2);
}

// Whether an output may be off because its activations' terms left their
// range: infinite or NaN, or so small (below 2^-90, but not zero) that what three
// bf16 terms cut off an activation, less than their last bit 2^-133 of it, could
// count.  An output of activations all below 2^-133 comes out zero.
// term_range is past kTermRange for all of these, and for zero.
constexpr uint32_t kTermLeast = (127u - 90u) << 24, kTermRange = 0xFEFFFFFFu - kTermLeast;

__device__ __forceinline__ uint32_t term_range(float v) { return (__float_as_uint(v) << 1) - kTermLeast; }

__device__ __forceinline__ bool out_of_terms(float v) { return v != 0.0f && term_range(v) > kTermRange; }

// Eight weights as their bf16 terms: one (bf16), or two (binary16).
template <bool HALF>
__device__ __forceinline__ void weight_terms(const uint4_t w, bf8_t (&t)[HALF ? 2 : 1]) {
  if constexpr (HALF) {
    uint4_t p0, p1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const half2_t h = as_half2(w[i]);
      const float a = (float)h.x, b = (float)h.y;
      p0[i] = high_pair(a, b);
      p1[i] = high_pair(a - high_part(a), b - high_part(b));
    }
    t[0] = __builtin_bit_cast(bf8_t, p0);
    t[1] = __builtin_bit_cast(bf8_t, p1);
  } else {
    t[0] = __builtin_bit_cast(bf8_t, w);
  }
}

// One output by fp32 FMAs over the row; a NaN stays one, so it ends the row.
template <bool HALF>
__device__ __forceinline__ float plain_dot(const float *x, const uint16_t *w, int K) {
  float sum = 0.0f;
  for (int k = 0; k < K && sum == sum; ++k) {
    const float v = HALF ? (float)__builtin_bit_cast(_Float16, w[k]) : __uint_as_float((uint32_t)w[k] << 16);
    sum = __builtin_fmaf(v, x[k], sum);
  }
  return sum;
}

template <int WN, int WM, int KS, int NB, int MB, int STAGES, bool HALF>
__global__ __launch_bounds__(64 * WN * WM * KS, WN * WM * KS <= 4 ? 2 : WN * WM * KS / 4) void gemm_real_kernel(GemmRealArgs g) {
  using F = RealForm<WN, WM, KS, NB, MB, STAGES>;
  constexpr int W = F::W, TN = F::TN, TM = F::TM;
  constexpr int WT = HALF ? 2 : 1;
  constexpr int kChain = 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = (wave / WN) % WM, ks = wave / (WN * WM);
  int tile_x, tile_y;
  xcd_tile(tile_x, tile_y);
  const int n0 = tile_x * TN, m0 = tile_y * TM;
  const int steps = (g.K + kRealStep * KS - 1) / (kRealStep * KS);
  const int gq = lane >> 4;  // lane group: k 8 gq .. 8 gq + 7 of a step
  const int n = lane & 15;

  // DMA sources at step 0.  Activations: 16-byte chunk f of a stage is step
  // f / (8 TM), row (f / 8) % TM, physical chunk f % 8 holding logical chunk
  // (f % 8) ^ ((row >> 1) & 7).  Weights: step f / (4 TN), row (f / 4) % TN,
  // logical chunk (f % 4) ^ ((row >> 2) & 3).  Either way the 16 rows a read
  // spans land in 16 distinct bank groups.  Rows past the tile's end read the
  // last row; a step past K (K not a whole number of stages) reads its row's
  // first step and is not multiplied.
  const float *a_src[F::NA];
  int a_in[F::NA];
#pragma unroll
  for (int u = 0; u < F::NA; ++u) {
    const int f = 64 * (wave + W * u) + lane;
    int kss = 0, row = 0, lc = 0;
    if (f < KS * TM * 8) {
      kss = f / (TM * 8);
      row = (f / 8) % TM;
      lc = (f & 7) ^ ((row >> 1) & 7);
    }
    a_src[u] = g.act + (size_t)min(m0 + row, g.M - 1) * (size_t)g.act_stride;
    a_in[u] = kss * kRealStep + 4 * lc;
  }
  const uint16_t *w_src[F::NW];
  int w_in[F::NW];
#pragma unroll
  for (int u = 0; u < F::NW; ++u) {
    const int f = 64 * (wave + W * u) + lane;
    int kss = 0, row = 0, lc = 0;
    if (f < KS * TN * 4) {
      kss = f / (TN * 4);
      row = (f / 4) % TN;
      lc = (f & 3) ^ ((row >> 2) & 3);
    }
    w_src[u] = g.rows + (size_t)min(n0 + row, g.N - 1) * (size_t)g.K;
    w_in[u] = kss * kRealStep + 8 * lc;
  }
  auto issue = [&](int s) {
    uint8_t *st = lds + (s % STAGES) * F::STAGE;
    const int k0 = s * (kRealStep * KS);
#pragma unroll
    for (int u = 0; u < F::NA; ++u) {
      const int k = k0 + a_in[u];
      __builtin_amdgcn_global_load_lds((real_global_t *)(a_src[u] + (KS == 1 || k < g.K ? k : 0)),
                                       (real_lds_t *)(st + 1024 * (wave + W * u)), 16, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < F::NW; ++u) {
      const int k = k0 + w_in[u];
      __builtin_amdgcn_global_load_lds((real_global_t *)(w_src[u] + (KS == 1 || k < g.K ? k : 0)),
                                       (real_lds_t *)(st + F::A_PAD + 1024 * (wave + W * u)), 16, 0, 0);
    }
  };

  // sum: the finished chains; small: every product of a term but the first;
  // chain: the first terms' products of kChain steps
  float4_t sum[MB][NB], small[MB][NB];
  const float4_t zero = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) sum[i][j] = small[i][j] = zero;

  // Software pipeline: STAGES - 1 steps in flight (a wait on this wave's
  // loads, then a bare barrier: a fence would wait for the later steps' too).
  constexpr int AHEAD = STAGES - 1;
  for (int t = 0; t < AHEAD && t < steps; ++t) issue(t);
  for (int s0 = 0; s0 < steps; s0 += kChain) {
    float4_t chain[MB][NB];
#pragma unroll
    for (int c = 0; c < kChain; ++c) {
      const int s = s0 + c;
      if (c > 0 && s >= steps) break;
      if (AHEAD >= 2 && s + AHEAD <= steps)
        real_wait<F::LOADS * (AHEAD - 1)>();
      else
        real_wait<0>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (s + AHEAD < steps) issue(s + AHEAD);
      if (KS > 1 && (s * KS + ks) * kRealStep >= g.K) {  // a step past K (wave-uniform)
        if (c == 0) {
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) chain[i][j] = zero;
        }
        continue;
      }
      const uint8_t *st = lds + (s % STAGES) * F::STAGE;
      bf8_t wt[NB][WT];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int row = (wn * NB + j) * 16 + n;
        weight_terms<HALF>(*reinterpret_cast<const uint4_t *>(st + F::A_PAD + (size_t)(ks * TN + row) * 64 +
                                                              16 * (gq ^ ((row >> 2) & 3))),
                           wt[j]);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int row = (wm * MB + i) * 16 + n;
        const uint8_t *at = st + (size_t)(ks * TM + row) * 128;
        const int sw = (row >> 1) & 7;
        bf8_t xa[3];
        split3(*reinterpret_cast<const float4_t *>(at + 16 * ((2 * gq) ^ sw)),
               *reinterpret_cast<const float4_t *>(at + 16 * ((2 * gq + 1) ^ sw)), xa);
#pragma unroll
        for (int t = 0; t <= 2 + WT - 1; ++t)  // the larger terms first: the smaller ones take longer to form
#pragma unroll
          for (int b = 0; b < WT; ++b) {
            const int a = t - b;
            if (a < 0 || a > 2) continue;
#pragma unroll
            for (int j = 0; j < NB; ++j) {
              if (t == 0)
                chain[i][j] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[0], wt[j][0], c == 0 ? zero : chain[i][j], 0, 0, 0);
              else
                small[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[a], wt[j][b], small[i][j], 0, 0, 0);
            }
          }
      }
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[i][j][r] += chain[i][j][r];
  }
  float4_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = sum[i][j][r] + small[i][j][r];

  // The K split's partial tiles, added in ks order.
  if (KS > 1) {
    __syncthreads();
    float *red = reinterpret_cast<float *>(lds);
    const int tile = wm * WN + wn;
    if (ks > 0) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            red[((((ks - 1) * WM * WN + tile) * MB * NB + i * NB + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int z = 1; z < KS; ++z)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][j][r] += red[((((z - 1) * WM * WN + tile) * MB * NB + i * NB + j) * 4 + r) * 64 + lane];
  }

  // A 16 x 16 tile of D: lane l holds lanes (C rows) 4 (l / 16) .. + 3 of
  // weight row (C column) l % 16.
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + (wm * MB + i) * 16 + 4 * gq + r;
      if (m >= g.M) continue;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int nn = n0 + (wn * NB + j) * 16 + n;
        if (nn >= g.N) continue;
        g.out[(size_t)m * (size_t)g.out_stride + nn] = acc[i][j][r];
      }
    }
  uint32_t worst = 0;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) worst = max(worst, term_range(acc[i][j][r]));
  if (worst <= kTermRange) return;
  // Some to form again, one by one.
  uint32_t again = 0;
  static_assert(MB * NB * 4 <= 32, "a bit an output");
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (m0 + (wm * MB + i) * 16 + 4 * gq + r < g.M && n0 + (wn * NB + j) * 16 + n < g.N &&
            out_of_terms(acc[i][j][r]))
          again |= 1u << ((i * NB + j) * 4 + r);
  for (; again; again &= again - 1) {
    const int bit = __builtin_ctz(again), tile = bit / 4;
    const int m = m0 + (wm * MB + tile / NB) * 16 + 4 * gq + bit % 4;
    const int nn = n0 + (wn * NB + tile % NB) * 16 + n;
    g.out[(size_t)m * (size_t)g.out_stride + nn] =
        plain_dot<HALF>(g.act + (size_t)m * (size_t)g.act_stride, g.rows + (size_t)nn * (size_t)g.K, g.K);
  }
}

// ---- forms and their choice -----------------------------------------------

template <int WN, int WM, int KS, int NB, int MB, int STAGES, bool HALF>
static hipError_t real_launch(const GemmRealArgs &a, hipStream_t stream) {
  using F = RealForm<WN, WM, KS, NB, MB, STAGES>;
  const void *fn = reinterpret_cast<const void *>(&gemm_real_kernel<WN, WM, KS, NB, MB, STAGES, HALF>);
  static bool granted = false;  // the dynamic LDS a kernel asks for is granted once
  if (!granted) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, F::LDS);
    if (e != hipSuccess) return e;
    granted = true;
  }
  const dim3 grid((a.N + F::TN - 1) / F::TN, (a.M + F::TM - 1) / F::TM);
  hipLaunchKernelGGL((gemm_real_kernel<WN, WM, KS, NB, MB, STAGES, HALF>), grid, dim3(64 * F::W), (size_t)F::LDS,
                     stream, a);
  return hipGetLastError();
}

// A launch takes, of the tiles 16 x 16, 32 x 16, 32 x 32, 64 x 32 and 64 x 64
// (rows x lanes; K split four or eight ways inside the workgroup), the smallest
// whose grid one round of the 256 CUs holds, up to sixteen lanes also 32 x 16 in
// workgroups two a CU (280 of them at 8960 rows: 8.8 us, against 10.5 on 64 x
// 32); past one round of 64 x 64 the same tile with K unsplit, three workgroups
// a CU.  Replayed, us, bf16, the chosen form and the ones beside it:
//   2560 x 1536:  16 lanes 5.3 (32 x 16: 6.4), 48 lanes 6.8 (16 x 16 in two
//                 rounds 7.1, 32 x 32 7.9), 130 lanes 10.4 (32 x 32 13.8, 64 x
//                 64 14.5), 300 lanes 14.8 (64 x 32 19.5, unsplit 21.1), 500
//                 lanes 24.3 (64 x 64 split 28.7)
//   8960 x 1536:  32 lanes 11.1 (32 x 32 14.1, 64 x 64 15.8), 64 lanes 15.1
//                 (64 x 32 22.8), 300 lanes 36.2 (64 x 64 split 45.8)
struct RealShape {
  int tn, tm, per_cu;
};
constexpr RealShape kRealForms[] = {{16, 16, 1}, {32, 16, 1}, {32, 16, 2}, {32, 32, 1}, {64, 32, 1}, {64, 64, 1}};
constexpr int kRealWide = 6;  // 64 x 64, K unsplit

static int real_form(int M, int N) {
  for (int f = 0; f < kRealWide; ++f) {
    const RealShape &s = kRealForms[f];
    if (s.per_cu > 1 && M > s.tm) continue;
    if ((long)((N + s.tn - 1) / s.tn) * ((M + s.tm - 1) / s.tm) <= 256L * s.per_cu) return f;
  }
  return kRealWide;
}

template <bool HALF>
static hipError_t real_pick(const GemmRealArgs &a, hipStream_t stream) {
  switch (real_form(a.M, a.N)) {
    case 0: return real_launch<1, 1, 8, 1, 1, 3, HALF>(a, stream);
    case 1: return real_launch<1, 1, 8, 2, 1, 3, HALF>(a, stream);
    case 2: return real_launch<1, 1, 4, 2, 1, 4, HALF>(a, stream);
    case 3: return real_launch<1, 2, 8, 2, 1, 2, HALF>(a, stream);
    case 4: return real_launch<1, 2, 8, 4, 1, 2, HALF>(a, stream);
    case 5: return real_launch<1, 4, 4, 4, 1, 3, HALF>(a, stream);
    default: return real_launch<1, 4, 1, 4, 1, 4, HALF>(a, stream);
  }
}

}  // namespace igl

using namespace igl;

// From five lanes: gemv_real_kernel then takes its eight-lane form, with K in
// chunks (8960 x 1536: 18 us against 8.6; 2560 x 1536: 14 against 5.3).
extern "C" int igl_gemm_real_fits(int real_type, int lanes, int N, int K) {
  return (real_type == IGL_STORE_BF16 || real_type == IGL_STORE_F16) && lanes >= 5 && N >= 1 && K >= 32 &&
         K % 32 == 0;
}

extern "C" int igl_gemm_real_form(int lanes, int N) { return real_form(lanes, N); }

extern "C" hipError_t igl_launch_gemm_real(const void *rows, int real_type, const float *act, int act_stride,
                                           int lanes, float *out, int out_stride, int N, int K, hipStream_t stream) {
  if (!igl_gemm_real_fits(real_type, lanes, N, K) || (((uintptr_t)act) & 15u) || (((uintptr_t)rows) & 15u) ||
      (act_stride & 3))
    return hipErrorInvalidValue;
  GemmRealArgs a;
  a.act = act;
  a.act_stride = act_stride;
  a.rows = static_cast<const uint16_t *>(rows);
  a.out = out;
  a.out_stride = out_stride;
  a.M = lanes;
  a.N = N;
  a.K = K;
  return real_type == IGL_STORE_F16 ? real_pick<true>(a, stream) : real_pick<false>(a, stream);
}
