// igl_gemm_few.h - a 4-bit plane times a few dozen lanes of fp32 activations,
// gfx950 bf16 MFMA.
//
// C[m][n] = sum_g gain[n][g] * sum_{k in g} x[m][k] * (c[n][k] - 8)
// with the reference's arithmetic (kern_row_code_many, app_core.c:4075-4117):
// a 32-code unit's dot product, then its gain by one fp32 FMA.  Between the
// GEMV, whose sixteen lanes a launch read the plane again for the next
// sixteen, and the prefill GEMM, whose 64-lane tiles, activation pass and
// workspace pay from 64 lanes.
//
// An fp32 activation is three bf16 terms exactly (split3) and a code less its
// bias one, so every product is exact and nothing of the activations passes
// through memory first: no workspace, one launch.  A unit's three products
// are chained from zero, the smallest term first.  Activations whose terms or
// unit sums leave that range are formed again (few_dot).
//
// Tiling as gemm_real_kernel's: WN x WM x KS waves own TN x TM of C, K in LDS
// stages of KS units filled by the LDS DMA, wave group ks takes a stage's
// ks-th unit, the KS partial tiles added in ks order at the end.
#pragma once

#include "igl_gemm_real.h"

namespace igl {

struct GemmFewArgs {
  const float *act;  // 16-byte aligned, act_stride % 4 == 0
  int act_stride;
  const uint8_t *codes;  // rows 16-byte aligned
  long long row_stride;
  const float *gains;  // [N][gain_stride]
  int gain_stride;
  int group_shift;  // gain of 32-code unit u: u >> group_shift
  float *out;
  int out_stride;
  int M, N, K;  // K % 32 == 0
};

template <int WN, int WM, int KS, int NB, int MB, int STAGES>
struct FewForm {
  static constexpr int W = WN * WM * KS;
  static constexpr int TN = 16 * NB * WN;
  static constexpr int TM = 16 * MB * WM;
  static constexpr int A_PAD = real_round(KS * TM * 128, 1024 * W);
  static constexpr int C_PAD = real_round(KS * TN * 16, 1024 * W);
  static constexpr int G_PAD = real_round(KS * TN * 4, 256 * W);
  static constexpr int C_OFF = A_PAD;
  static constexpr int G_OFF = A_PAD + C_PAD;
  static constexpr int STAGE = G_OFF + G_PAD;
  static constexpr int RED = (KS - 1) * TN * TM * 4;
  static constexpr int LDS = STAGES * STAGE > RED ? STAGES * STAGE : RED;
  static constexpr int NA = A_PAD / (1024 * W);
  static constexpr int NC = C_PAD / (1024 * W);
  static constexpr int NG = G_PAD / (256 * W);
  static constexpr int LOADS = NA + NC + NG;
  static_assert(LDS <= 160 * 1024, "LDS");
  static_assert(LOADS * (STAGES - 2) < 64, "vmcnt");
};

// Eight codes (low nibble first) less 8 as bf16.
__device__ __forceinline__ bf8_t code_terms(uint32_t d) {
  const int v = (int)(d ^ 0x88888888u);
  uint4_t p;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    p[i] = high_pair((float)(v << (28 - 8 * i) >> 28), (float)(v << (24 - 8 * i) >> 28));
  return __builtin_bit_cast(bf8_t, p);
}

// One output by fp32 FMAs, where out_of_terms(v) says that the terms may not
// have held it.  Past fp32's range (an infinite or NaN activation, or finite
// ones whose unit's sum overflows before its gain) the gain goes in first; below,
// last, as a unit's sum of subnormal activations is exact.  A NaN stays one, so
// it ends the row.  The check of a tile's outputs is within the runs' noise (6144
// x 1536 at 37 lanes 13.1 us, 13.1 without); one output's bits each, gathered as
// it is stored, cost 0.5 us.
__device__ __forceinline__ float few_dot(const float *x, const uint8_t *codes, const float *gains,
                                         int group_shift, int units, float v) {
  const bool below = fabsf(v) < 1.0f;
  float sum = 0.0f;
  for (int u = 0; u < units && sum == sum; ++u) {
    const float gain = gains[u >> group_shift];
    const float first = below ? 1.0f : gain, last = below ? gain : 1.0f;
    const uint4_t c = *reinterpret_cast<const uint4_t *>(codes + 16 * u);
    float dot = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float4_t a = *reinterpret_cast<const float4_t *>(x + 32 * u + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int code = (int)((c[i / 2] >> (16 * (i & 1) + 4 * e)) & 15u) - 8;
        dot = __builtin_fmaf((float)code * first, a[e], dot);
      }
    }
    sum = __builtin_fmaf(last, dot, sum);
  }
  return sum;
}

template <int WN, int WM, int KS, int NB, int MB, int STAGES>
__global__ __launch_bounds__(64 * WN * WM * KS, WN * WM * KS <= 4 ? 2 : WN * WM * KS / 4) void gemm_few_kernel(
    GemmFewArgs g) {
  using F = FewForm<WN, WM, KS, NB, MB, STAGES>;
  constexpr int W = F::W, TN = F::TN, TM = F::TM;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = (wave / WN) % WM, ks = wave / (WN * WM);
  int tile_x, tile_y;
  xcd_tile(tile_x, tile_y);
  const int n0 = tile_x * TN, m0 = tile_y * TM;
  const int units = g.K / 32;
  const int steps = (units + KS - 1) / KS;
  const int gq = lane >> 4;  // lane group: k 8 gq .. 8 gq + 7 of a unit
  const int n = lane & 15;

  // DMA sources at step 0, rows past the end the last row, units past K the
  // row's first (not multiplied).  Activations as gemm_real_kernel's: unit f /
  // (8 TM), row (f / 8) % TM, physical chunk f % 8 holding chunk (f % 8) ^ ((row
  // >> 1) & 7).  Codes: row f / KS, physical slot f % KS holding unit (f % KS) ^
  // (row % KS), so a row's KS units are one run of memory and the 16 rows of a
  // read spread over the banks.  Gains: row f / KS, unit f % KS.
  const float *a_src[F::NA];
  int a_unit[F::NA];
#pragma unroll
  for (int u = 0; u < F::NA; ++u) {
    const int f = 64 * (wave + W * u) + lane;
    int kss = 0, row = 0, lc = 0;
    if (f < KS * TM * 8) {
      kss = f / (TM * 8);
      row = (f / 8) % TM;
      lc = (f & 7) ^ ((row >> 1) & 7);
    }
    a_src[u] = g.act + (size_t)min(m0 + row, g.M - 1) * (size_t)g.act_stride + 4 * lc;
    a_unit[u] = kss;
  }
  const uint8_t *c_src[F::NC];
  int c_unit[F::NC];
#pragma unroll
  for (int u = 0; u < F::NC; ++u) {
    const int f = 64 * (wave + W * u) + lane;
    int kss = 0, row = 0;
    if (f < KS * TN) {
      row = f / KS;
      kss = (f % KS) ^ (row % KS);
    }
    c_src[u] = g.codes + (size_t)min(n0 + row, g.N - 1) * (size_t)g.row_stride;
    c_unit[u] = kss;
  }
  const float *g_src[F::NG];
  int g_unit[F::NG];
#pragma unroll
  for (int u = 0; u < F::NG; ++u) {
    const int f = 64 * (wave + W * u) + lane;
    int kss = 0, row = 0;
    if (f < KS * TN) {
      row = f / KS;
      kss = f % KS;
    }
    g_src[u] = g.gains + (size_t)min(n0 + row, g.N - 1) * (size_t)g.gain_stride;
    g_unit[u] = kss;
  }
  auto issue = [&](int s) {
    uint8_t *st = lds + (s % STAGES) * F::STAGE;
    const int u0 = s * KS;
#pragma unroll
    for (int u = 0; u < F::NA; ++u) {
      const int at = u0 + a_unit[u];
      __builtin_amdgcn_global_load_lds((real_global_t *)(a_src[u] + 32 * (at < units ? at : 0)),
                                       (real_lds_t *)(st + 1024 * (wave + W * u)), 16, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < F::NC; ++u) {
      const int at = u0 + c_unit[u];
      __builtin_amdgcn_global_load_lds((real_global_t *)(c_src[u] + 16 * (at < units ? at : 0)),
                                       (real_lds_t *)(st + F::C_OFF + 1024 * (wave + W * u)), 16, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < F::NG; ++u) {
      const int at = u0 + g_unit[u];
      __builtin_amdgcn_global_load_lds((real_global_t *)(g_src[u] + ((at < units ? at : 0) >> g.group_shift)),
                                       (real_lds_t *)(st + F::G_OFF + 256 * (wave + W * u)), 4, 0, 0);
    }
  };

  // acc: the last kRun steps' units; sum: the runs before
  constexpr int kRun = 8;
  float4_t acc[MB][NB], sum[MB][NB];
  const float4_t zero = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = sum[i][j] = zero;

  // Software pipeline: STAGES - 1 steps in flight (a wait on this wave's
  // loads, then a bare barrier: a fence would wait for the later steps' too).
  constexpr int AHEAD = STAGES - 1;
  for (int t = 0; t < AHEAD && t < steps; ++t) issue(t);
  for (int s = 0; s < steps; ++s) {
    if (AHEAD >= 2 && s + AHEAD <= steps)
      real_wait<F::LOADS * (AHEAD - 1)>();
    else
      real_wait<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + AHEAD < steps) issue(s + AHEAD);
    if (s % kRun == 0 && s > 0) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
#pragma unroll
          for (int r = 0; r < 4; ++r) sum[i][j][r] += acc[i][j][r];
          acc[i][j] = zero;
        }
    }
    if (KS > 1 && s * KS + ks >= units) continue;  // a unit past K (wave-uniform)
    const uint8_t *st = lds + (s % STAGES) * F::STAGE;
    bf8_t wt[NB];
    float gain[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int row = (wn * NB + j) * 16 + n;
      wt[j] = code_terms(
          *reinterpret_cast<const uint32_t *>(st + F::C_OFF + 16 * (row * KS + (ks ^ (row % KS))) + 4 * gq));
      gain[j] = *reinterpret_cast<const float *>(st + F::G_OFF + 4 * (row * KS + ks));
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int row = (wm * MB + i) * 16 + n;
      const uint8_t *at = st + (size_t)(ks * TM + row) * 128;
      const int sw = (row >> 1) & 7;
      bf8_t xa[3];
      split3(*reinterpret_cast<const float4_t *>(at + 16 * ((2 * gq) ^ sw)),
             *reinterpret_cast<const float4_t *>(at + 16 * ((2 * gq + 1) ^ sw)), xa);
      float4_t p[NB];
#pragma unroll
      for (int t = 2; t >= 0; --t)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          p[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[t], wt[j], t == 2 ? zero : p[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(gain[j], p[j][r], acc[i][j][r]);
    }
  }

#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] += sum[i][j][r];

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
    float *out = g.out + (size_t)m * (size_t)g.out_stride + nn;
    *out = few_dot(g.act + (size_t)m * (size_t)g.act_stride, g.codes + (size_t)nn * (size_t)g.row_stride,
                   g.gains + (size_t)nn * (size_t)g.gain_stride, g.group_shift, units, *out);
  }
}

// ---- forms and their choice -----------------------------------------------

template <int WN, int WM, int KS, int NB, int MB, int STAGES>
static hipError_t few_launch(const GemmFewArgs &a, hipStream_t stream) {
  using F = FewForm<WN, WM, KS, NB, MB, STAGES>;
  const void *fn = reinterpret_cast<const void *>(&gemm_few_kernel<WN, WM, KS, NB, MB, STAGES>);
  static bool granted = false;  // the dynamic LDS a kernel asks for is granted once
  if (!granted) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, F::LDS);
    if (e != hipSuccess) return e;
    granted = true;
  }
  const dim3 grid((a.N + F::TN - 1) / F::TN, (a.M + F::TM - 1) / F::TM);
  hipLaunchKernelGGL((gemm_few_kernel<WN, WM, KS, NB, MB, STAGES>), grid, dim3(64 * F::W), (size_t)F::LDS, stream, a);
  return hipGetLastError();
}

// The tiles (weight rows x lanes, K split sixteen ways inside the workgroup in
// the first two, eight in the others, four in 64 x 64) in the order a launch
// tries them; it takes the first whose grid its rounds hold.  Replayed, us, the chosen form against its neighbours:
//   6144 x 1536: 24 lanes 48 x 16 8.1 (32 x 32 10.0, 64 x 32 13.9), 37 lanes 32 x
//                48 12.6 (64 x 32 14.6), 63 lanes 48 x 16 11.6 (64 x 32 14.7)
//   1536 x 6144: 24 lanes 16 x 16 13.8 (32 x 16 17.9), 63 lanes 32 x 16 18.4 (16 x
//                16 25.5, 32 x 32 28.1)
//   8192 x 8192: 24 lanes 32 x 32 37.5 (48 x 16 43.3), 37 lanes 32 x 48 48.4 (64 x
//                32 57.6), 63 lanes 64 x 32 58.4 (48 x 16 64.9)
//   12288 x 2048, 63 lanes: 64 x 64 28.3 (64 x 32 in two rounds 32.4)
struct FewShape {
  int tn, tm, wgs;  // wgs: workgroups the grid may have
};
constexpr FewShape kFewForms[] = {{16, 16, 256}, {32, 16, 256}, {48, 16, 256}, {32, 32, 256},
                                  {32, 48, 256}, {48, 16, 512}, {64, 32, 256}};
constexpr int kFewWide = 7;  // 64 x 64

static int few_form(int M, int N) {
  for (int f = 0; f < kFewWide; ++f) {
    const FewShape &s = kFewForms[f];
    if ((long)((N + s.tn - 1) / s.tn) * ((M + s.tm - 1) / s.tm) <= s.wgs) return f;
  }
  return kFewWide;
}

}  // namespace igl

using namespace igl;

// From seventeen lanes, where the GEMV reads the plane again for every sixteen
// (37 lanes, us: 6144 x 1536 34.5 -> 12.6, 1536 x 6144 29.5 -> 17.8, 8192 x 8192
// 117 -> 48); from nine but on few long rows, which the GEMV cuts into K-chunks
// of workgroups (12 lanes: 6144 x 1536 13.3 -> 7.4, 8192 x 8192 46 -> 24, but 1536 x
// 6144 10.4 against 13.2, 256 x 4096 7.2 against 9.5).  To 63 lanes; from 64 the
// prefill GEMM.
extern "C" int igl_gemm_few_fits(int lanes, int N, int K) {
  return N >= 1 && K >= 32 && K % 32 == 0 && lanes <= 63 &&
         (lanes >= 17 || (lanes >= 9 && (K < 4096 || N >= 4096)));
}

extern "C" int igl_gemm_few_form(int lanes, int N) { return few_form(lanes, N); }

// Arguments as igl_launch_gemv_q4's (code bias 8), activations 16-byte aligned
// with act_stride % 4 == 0, no workspace.
extern "C" hipError_t igl_launch_gemm_few(const uint8_t *codes, long long row_stride, const float *gains,
                                          int gain_stride, int group_shift, const float *act, int act_stride, int lanes,
                                          float *out, int out_stride, int N, int K, hipStream_t stream) {
  if (!igl_gemm_few_fits(lanes, N, K) || (((uintptr_t)act) & 15u) || (act_stride & 3) || (((uintptr_t)codes) & 15u) ||
      (row_stride & 15))
    return hipErrorInvalidValue;
  GemmFewArgs a;
  a.act = act;
  a.act_stride = act_stride;
  a.codes = codes;
  a.row_stride = row_stride;
  a.gains = gains;
  a.gain_stride = gain_stride;
  a.group_shift = group_shift;
  a.out = out;
  a.out_stride = out_stride;
  a.M = lanes;
  a.N = N;
  a.K = K;
  switch (few_form(lanes, N)) {
    case 0: return few_launch<1, 1, 16, 1, 1, 2>(a, stream);
    case 1: return few_launch<1, 1, 16, 2, 1, 3>(a, stream);
    case 2:
    case 5: return few_launch<1, 1, 8, 3, 1, 3>(a, stream);
    case 3: return few_launch<1, 1, 8, 2, 2, 3>(a, stream);
    case 4: return few_launch<1, 1, 8, 2, 3, 2>(a, stream);
    case 6: return few_launch<1, 2, 8, 4, 1, 3>(a, stream);
    default: return few_launch<1, 4, 4, 4, 1, 3>(a, stream);
  }
}
