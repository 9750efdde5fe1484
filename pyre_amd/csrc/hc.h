// What the launches of a hyper-connection mix share (hc.hip, hc_cols.hip, hc_m.hip).
#pragma once
#include "formats.h"

__device__ __forceinline__ float sigm(float x) { return 1.0f / (1.0f + expf(-x)); }

// Stream element i of token ti with the pending residual update applied: x + out * w  (:1384-1387), w = 2*sigm(inj).
// `out` is a plain [t][d] vector (comb_out) or the unreduced FFN output (mo.partial != nullptr).
// NP > 1: `out` comes as NP partial vectors, part q of token ti at comb_out + (q*T + ti)*d, added in order from the first
// (pyre_gemv_parts_launch); all parts are fetched before the first add.  NP = 0: never unreduced.
template <int T, int NP, int FK = 0, int FG = 0> __device__ __forceinline__ float hc_x_new(const float* __restrict__ x_in, int in_ss, int in_ts, const float* __restrict__ comb_out, const MoeOut& mo, float w, int d, int ti, int s, int i) {
  float v = x_in[(size_t)ti * in_ts + (size_t)s * in_ss + i];
  if constexpr (NP > 1) {
    float sv[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) sv[q] = (comb_out + ((size_t)q * T + ti) * d)[i];
    float o = sv[0];
#pragma unroll
    for (int q = 1; q < NP; ++q) o += sv[q];
    v = v + o * w;
  } else {
    if (NP == 1 && mo.partial) v = v + moe_out_value<FK, FG>(mo, ti, i) * w;
    else if (comb_out) v = v + comb_out[(size_t)ti * d + i] * w;
  }
  return v;
}

// x / n for 0 <= x < 2^16, n <= 2^12 with r = 1 / n within two units in the last place: (x + 1/2) / n lies 1 / (2 n) or more off an
// integer, the product's error is below x / n * 2^-21
__device__ __forceinline__ int hc_div(int x, float r) { return (int)(((float)x + 0.5f) * r); }
__device__ __forceinline__ float hc_recip(int n) { return __builtin_amdgcn_rcpf((float)n); }
// v / hc; a power of two by multiplication, the same bits
__device__ __forceinline__ float hc_mean(float v, int hc) { return (hc & (hc - 1)) == 0 ? v * __uint_as_float((uint32_t)(127 - (31 - __builtin_clz(hc))) << 23) : v / (float)hc; }

// The slices of one output row, all loads in flight together: groups of eight behind a branch the whole launch agrees on
// (ksplit is a kernel argument), so that unused groups cost neither loads nor instruction fetch; inside a group slices
// past ksplit repeat the last one and are never added.  `want` is the thread's own condition (one execution mask).
template <int KSM> __device__ __forceinline__ void hc_load_run(float (&sv)[KSM], const float* __restrict__ p, int n, int stride) {      // n (<= KSM) values at p, p + stride, ..
#pragma unroll
  for (int k = 0; k < KSM; ++k) sv[k] = 0.0f;
#pragma unroll
  for (int g = 0; g < KSM / 4; ++g) if (g * 4 < n) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sv[g * 4 + j] = p[(size_t)min(g * 4 + j, n - 1) * stride];
  }
}
template <int T, int KSM> __device__ __forceinline__ void hc_load_slices(float (&pv)[KSM], const float* __restrict__ part, bool want, int ksplit, int t, int r64, int i) {
#pragma unroll
  for (int ks = 0; ks < KSM; ++ks) pv[ks] = 0.0f;
  const unsigned off = (unsigned)(t * r64 + i);
  if (want) {
#pragma unroll
    for (int g = 0; g < KSM / 8; ++g) if (g * 8 < ksplit) {
#pragma unroll
      for (int j = 0; j < 8; ++j) pv[g * 8 + j] = (part + (size_t)min(g * 8 + j, ksplit - 1) * T * r64)[off];      // launch-uniform base + the thread's 32-bit offset
    }
  }
}

// the slices of one row in order, each times its stream's scale (sls: at least KSM floats); whole groups of four carry no predicates
template <int KSM> __device__ __forceinline__ float hc_slice_sum(const float (&pv)[KSM], const float* sls, int ksplit) {
  float o = 0.0f;
#pragma unroll
  for (int g = 0; g < KSM; g += 4) if (g < ksplit) {
    float sc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) sc[j] = sls[g + j];
    if (g + 4 <= ksplit) {
#pragma unroll
      for (int j = 0; j < 4; ++j) { const float tm = pv[g + j] * sc[j]; o = g + j == 0 ? tm : o + tm; }
    } else {
#pragma unroll
      for (int j = 0; j < 3; ++j) if (g + j < ksplit) { const float tm = pv[g + j] * sc[j]; o = g + j == 0 ? tm : o + tm; }
    }
  }
  return o;
}
// the gate logit: U (<= 16) sums `stride` floats apart in order, four in flight at a time
__device__ __forceinline__ float hc_unit_sum(const float* red, int U, int stride) {
  float g = red[0];
#pragma unroll
  for (int k = 1; k < 16; k += 3) if (k < U) {
    float v[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = red[min(k + j, U - 1) * stride];
#pragma unroll
    for (int j = 0; j < 3; ++j) if (k + j < U) g += v[j];
  }
  return g;
}

// the mixes whose straight code the smaller bounds hold: up to four streams of up to sixteen slices in all
inline bool pyre_hc_few(const HcDev& h, int ksplit) { return h.hc <= 4 && ksplit <= 16; }
int pyre_hc_up_cols_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, int t, const float* xnew, float eps, float* mixed, float* inj);

// the mixes on the matrix cores (hc_m.hip): whether a mix is one, the slices of its first launch, the two launches
bool pyre_hc_on_matrix_cores(const HcDev& h);
int pyre_hc_m_slices(const HcDev& h);
int pyre_hc_norm_down_m_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, const float* x_in, int in_ss, int in_ts, float* x_out, int t, const float* comb_out, int comb_parts, const MoeOut& mo, const float* comb_inj);
int pyre_hc_up_mix_m_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, int t, const float* xnew, float eps, float* mixed, float* inj, const HcRoute* rt, const AopOut* aop);
