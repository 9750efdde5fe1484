// Hyper-connection mix / combine around every block: grouped RMSNorm over the hc residual streams, low-rank sigmoid
// gate, stream mean; residual update.  Follows hc_mix / hc_combine, src/model/qwen4exp_gguf.rs:1357-1388 (f32 branch).
//
// One mix is two launches.  k_hc_norm_down folds the pending residual update, the norm weights and the [down ; inject]
// GEMV (K cut into slices, one slice per workgroup) and leaves each slice's sum of squares; k_hc_up_mix turns those
// into the streams' RMS scales, adds the scaled slice sums, applies silu, runs the up GEMV from shared memory and
// reduces the gated, normalized streams to their mean.  Mixes on the matrix cores: hc_m.hip; the second launch of windows in some
// formats: hc_cols.hip.
#include "hc.h"
#include <stdlib.h>
#include <algorithm>

PYRE_TS_DECL(hc_ts) PYRE_TS_EXPORT(hc_ts, pyre_debug_ts_hc)

// A unit of a matrix against T tokens in shared memory, rows of xstride floats: from PYRE_MMA_MIN tokens on by the matrix cores (the same bits), which
// read a unit's activations with one 16-byte load a lane and four tokens where the multiply-adds read every one for every lane.  HC_PAD: the four tokens
// a wave reads at a time meet four different sets of banks.  200 tokens of A3B's shape, bf16, groups of eight, us: first launch 47 -> 43, second 40 -> 33, with
// the router 60 -> 42.
#define HC_PAD 16
template <int FMT, int T> __device__ __forceinline__ void hc_unit(const QMatDev& m, const UnitRaw<FMT>& r, int ku, int lane, const float* xs, int xstride, float (&acc)[T]) {
  if constexpr (T < PYRE_MMA_MIN) { const uint2* lds2 = nullptr; unit_fma<FMT, T>(m, r, ku, lds2, lane, xs, xstride, acc); }
  else {
    constexpr int NG = (T + 3) / 4; XGrp<NG> x; v4f a[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const float4 v = *(const float4*)(xs + min(4 * g + (lane & 3), T - 1) * xstride + 4 * (lane >> 2)); x.x[g] = f4u{v.x, v.y, v.z, v.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) a[g][t] = 4 * g + t < T ? acc[4 * g + t < T ? 4 * g + t : 0] : 0.0f;
    }
    unit_mma<FMT, NG>(m, r, ku, x, a);
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = a[t >> 2][t & 3];
  }
}
// grid (row tiles of [down ; inject], K slices of a stream, streams x groups of tokens), nw waves.  A workgroup owns L = nw*upw*64 columns
// of one stream s.
// The RMS scale of a stream multiplies every term of a row's dot product, so it is applied after the dot (by
// k_hc_up_mix, which also sums the slices): a workgroup never needs the sum of squares of the whole stream.
//   1. its L columns of x_new (the pending residual update applied) times the norm weight go to shared memory; the
//      squares of x_new are summed over the slice -> ssq[ks*T + t]; the tile-0 workgroup of the slice also publishes the
//      updated stream (x_out, never the buffer x_in points into)
//   2. each wave takes upw units of the slice; partial sums -> part[(ks*T + t)*tiles*64 + row]
// ONE: eight waves of one unit each (every width in multiples of 512 with at most 32 slices): a thread prepares one column and a wave
// forms one unit's sums, without loops.  FG > 0: the experts a group of the unreduced FFN output (moe_out_value).  One token, bf16,
// 2048 columns, 6.1 us with the loops and the groups at run time, 5.0 with neither; 500 tokens' groups of eight 218 and 113 us.
// ALLT (groups of eight of a longer prompt): one workgroup for all row tiles, which otherwise prepare the same columns each: 200 tokens 43 -> 26 us.
template <int FMT, int T, int NP, bool ONE = false, int FG = 0, bool ALLT = false> __global__ __launch_bounds__(512) void k_hc_norm_down(QMatDev m, const float* __restrict__ x_in, int in_ss, int in_ts, float* __restrict__ x_out,
    const float* __restrict__ comb_out, MoeOut mo, const float* __restrict__ comb_inj, const float* __restrict__ norm, int d, int hc, float* __restrict__ ssq,
    float* __restrict__ part, int upw, const uint2* __restrict__ g2) {
  int s = blockIdx.z;
  if (s >= hc) {          // a further group of T tokens (pyre_hc_mix_rows_launch)
    const int grp = s / hc, ksplit = gridDim.y * hc; s -= grp * hc;
    const size_t zt = (size_t)grp * T;
    if (mo.partial) { mo.partial += zt * (mo.k + 1) * mo.d; mo.sel_w += zt * mo.k; mo.sg += zt; }
    x_in += zt * in_ts; x_out += zt * hc * d; ssq += zt * ksplit; part += zt * ksplit * ((size_t)m.tiles * 64);
    if (comb_out) comb_out += zt * d;
    if (comb_inj) comb_inj += zt * hc;
  }
  PYRE_TS_VARS PYRE_TS(0);
  qmat_args_now(m); args_now(x_in, in_ss, in_ts, x_out, comb_out, mo.partial, mo.sel_w, mo.sg, mo.d, mo.k, comb_inj, norm, d, hc, ssq, part, upw);
  if constexpr (ONE) upw = 1;
  extern __shared__ __align__(16) float sm[];
  const int nthr = ONE ? 512 : blockDim.x, nw = nthr >> 6, tid = threadIdx.x, L = nw * upw * 64, LP = L + HC_PAD;
  float* xs = sm;                         // [T][LP]
  float* red = sm + (size_t)T * LP;       // [nw][T][64], ALLT: twice
  float* wsum = red + (ALLT ? 2 : 1) * (size_t)nw * T * 64;   // [nw][T]
  const int tile = ALLT ? 0 : blockIdx.x, ks = s * gridDim.y + blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int i0 = blockIdx.y * L;
  // Loads return in the order they were issued: the streams (and the pending update's terms) first, since the copy into
  // shared memory waits for them, then the first unit's weights, which stay in flight across the barrier.
  float w[T], ss[T];
#pragma unroll
  for (int t = 0; t < T; ++t) { w[t] = (comb_out || mo.partial) ? 2.0f * sigm(comb_inj[t * hc + s]) : 0.0f; ss[t] = 0.0f; }
  float v0[T]; float nv0 = 0.0f;
  if (tid < L) {
    nv0 = norm[(size_t)s * d + i0 + tid];
#pragma unroll
    for (int t = 0; t < T; ++t) v0[t] = hc_x_new<T, NP, 0, FG>(x_in, in_ss, in_ts, comb_out, mo, w[t], d, t, s, i0 + tid);
  }
  UnitRaw<FMT> raw = unit_load<FMT>(m, tile, ks * nw * upw + wave * upw, lane);
  if (tid < L) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const float v = v0[t];
      ss[t] += v * v;
      xs[(size_t)t * LP + tid] = v * nv0;
      if (tile == 0) x_out[((size_t)t * hc + s) * d + i0 + tid] = v;
    }
  }
  if constexpr (!ONE) for (int j = tid + nthr; j < L; j += nthr) {
    const float nv = norm[(size_t)s * d + i0 + j];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float v = hc_x_new<T, NP>(x_in, in_ss, in_ts, comb_out, mo, w[t], d, t, s, i0 + j);
      ss[t] += v * v;
      xs[(size_t)t * LP + j] = v * nv;
      if (tile == 0) x_out[((size_t)t * hc + s) * d + i0 + j] = v;
    }
  }
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss[t] += __shfl_xor(ss[t], o);
    if (lane == 0) wsum[wave * T + t] = ss[t];
  }
  lds_barrier(); PYRE_TS(1);
  if (tile == 0 && tid < T) { float tot = wsum[tid]; for (int q = 1; q < nw; ++q) tot += wsum[q * T + tid]; ssq[ks * T + tid] = tot; }
  const size_t r64 = (size_t)m.tiles * 64;
  float acc[T];
  if constexpr (ALLT) {          // every row tile, the next one's weights in flight, the waves' sums of two tiles taking turns in shared memory
    static_assert(ONE, "a unit a wave");
    for (int tl = 0; tl < m.tiles; ++tl) {
      const UnitRaw<FMT> r = raw; float* rd = red + (size_t)(tl & 1) * nw * T * 64;
      raw = unit_load<FMT>(m, min(tl + 1, m.tiles - 1), ks * nw + wave, lane);
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t] = 0.0f;
      hc_unit<FMT, T>(m, r, ks * nw + wave, lane, xs + wave * 64, LP, acc);
#pragma unroll
      for (int t = 0; t < T; ++t) rd[((size_t)wave * T + t) * 64 + lane] = acc[t];
      lds_barrier();
      for (int i = tid; i < T * 64; i += nthr) {
        const int t = i >> 6, l = i & 63; float a = rd[(size_t)t * 64 + l];
        for (int q = 1; q < nw; ++q) a += rd[((size_t)q * T + t) * 64 + l];
        part[((size_t)ks * T + t) * r64 + (size_t)tl * 64 + l] = a;
      }
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = 0.0f;
  for (int u = 0; u < upw; ++u) { int lu = wave * upw + u; if (u > 0) raw = unit_load<FMT>(m, tile, ks * nw * upw + lu, lane); hc_unit<FMT, T>(m, raw, ks * nw * upw + lu, lane, xs + lu * 64, LP, acc); }
#pragma unroll
  for (int t = 0; t < T; ++t) red[((size_t)wave * T + t) * 64 + lane] = acc[t];
  PYRE_TS(2);
  lds_barrier(); PYRE_TS(3);
  for (int i = tid; i < T * 64; i += nthr) {
    int t = i >> 6, l = i & 63; float a = red[(size_t)t * 64 + l];
    for (int q = 1; q < nw; ++q) a += red[((size_t)q * T + t) * 64 + l];
    part[((size_t)ks * T + t) * r64 + (size_t)tile * 64 + l] = a;
  }
  PYRE_TS(4); PYRE_TS_FLUSH(hc_ts, NP > 1 ? 0 : 8);
}

// grid (d / 64), hc*U waves (U = lr / 64 units of the up matrix).  Prologue: the streams' RMS scales from the slice
// sums of squares, scale_s = 1 / sqrt(sum / d + eps) (rms, :209); o = the slice sums of [down ; inject], each times
// its stream's scale, added in slice order;
// lo = silu(o / hc) for the first lr rows -> shared memory, inj = o[lr + s] / hc (zeros without inject) (:1376-1378).
// Wave (s, ku) takes unit ku of row tile s*(d/64) + blockIdx.x of `up`; the gate logit of stream s is the sum of its
// waves in unit order; mixed[i] = (sum_s xn[s][i] * sigm(gate_s[i])) / hc with xn = (x * scale_s) * norm, s ascending
// from zero (:1380).
// RF >= 0: the launch also leaves its K slice of the router GEMV over the mixed vector (format RF; HcRoute): wave w
// takes router tile w, w + nw, .. at unit blockIdx.x, the first tile's weights fetched ahead of the up GEMV.
// KSM, HM: bounds of the slice and stream counts, which size the straight code (the launcher takes the smallest that holds the mix).
// FLR > 0: a low rank of FLR and exactly KSM slices, at compile time.
template <int FMT, int T, int RF, int KSM, int HM, int FLR = 0> __global__ __launch_bounds__(1024) void k_hc_up_mix(QMatDev up, const float* __restrict__ part, const float* __restrict__ ssq, int ksplit, int r64, int lr, int hc, int has_inject,
    const float* __restrict__ xnew, const float* __restrict__ norm, float eps, int d, float* __restrict__ mixed, float* __restrict__ inj, const uint2* __restrict__ g2,
    QMatDev router, float* __restrict__ rpart) {
  constexpr bool ROUTE = RF >= 0; constexpr int RFX = ROUTE ? RF : FMT_F32;
  if constexpr (FLR > 0) { lr = FLR; ksplit = KSM; }
  if (blockIdx.z) {          // a further group of T tokens (pyre_hc_mix_rows_launch)
    const size_t z = blockIdx.z; part += z * ksplit * T * r64; ssq += z * ksplit * T; xnew += z * T * hc * d; mixed += z * T * d; inj += z * T * hc;
    if (ROUTE) rpart += z * (d / 64) * T * router.tiles * 64;
  }
  const uint2* lds2 = nullptr;          // no format needs a codebook in shared memory any more
  PYRE_TS_VARS PYRE_TS(0);
  qmat_args_now(up); args_now(part, ssq, ksplit, r64, lr, hc, has_inject, xnew, norm, eps, d, mixed, inj);

  extern __shared__ __align__(16) float sm[];
  const int tid = threadIdx.x, U = lr >> 6, nthr = hc * lr, nw = hc * U;
  const float rhc = hc_recip(hc); const int kps = __builtin_amdgcn_readfirstlane(hc_div(ksplit, rhc));
  const int LP = lr + HC_PAD;
  float* lo = sm;                         // [T][LP]
  float* red = sm + (size_t)T * LP;       // [nw][T][64]
  float* sls = red + (size_t)nw * T * 64;   // [T][32]: the RMS scale of the stream each slice belongs to
  float* term = sls + (size_t)T * 32;     // [T*hc][64]: the streams' gated, normalized values before they are added
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int s = __builtin_amdgcn_readfirstlane(hc_div(wave, hc_recip(U))), ku = wave - s * U;
  // Loads return in the order they were issued, so they are issued in the order they are needed: the slice sums of
  // squares and of [down ; inject] first (the prologue waits for nothing else), then the up weights, the epilogue's
  // operands and the router tile, all of which stay in flight across the barriers below (which exchange through shared
  // memory only).
  float ssv[KSM];
#pragma unroll
  for (int k = 0; k < KSM; ++k) ssv[k] = 0.0f;
  const int stt = hc_div(tid, rhc), sq = tid - stt * hc;
  if (tid < T * hc) hc_load_run<KSM>(ssv, ssq + (size_t)(sq * kps) * T + stt, kps, T);          // all of the stream's slices before the first add: one round trip
  // the slices of rows of lo, with few slices two rounds of a row a thread ahead (T / hc rounds)
  constexpr bool AHEAD = KSM <= 16 && T > 1;
  const float rlr = hc_recip(lr); const int n_lo = T * lr;
  float pv[KSM], pn[AHEAD ? KSM : 1];
  auto slices = [&](float (&v)[KSM], int idx) { const int t = hc_div(idx, rlr); hc_load_slices<T, KSM>(v, part, idx < n_lo, ksplit, t, r64, idx - t * lr); };
  slices(pv, tid);
  if constexpr (AHEAD) { if (n_lo > nthr) slices(pn, tid + nthr); }
  constexpr bool U_EARLY = FMT != FMT_F32 || T == 1;      // an f32 unit is 64 registers: with several tokens' it waits for the slice sums'
  UnitRaw<FMT> raw;
  if constexpr (U_EARLY) raw = unit_load<FMT>(up, s * (d >> 6) + blockIdx.x, ku, lane);
  // the epilogue's stream value and norm weight of this wave's first (token, stream) item
  float xpre = 0.0f, npre = 0.0f;
  if (wave < T * hc) { const int t0 = __builtin_amdgcn_readfirstlane(hc_div(wave, rhc)), q0 = wave - t0 * hc; xpre = (xnew + ((size_t)t0 * hc + q0) * d + blockIdx.x * 64)[lane]; npre = (norm + (size_t)q0 * d + blockIdx.x * 64)[lane]; }
  UnitRaw<RFX> rraw;
  constexpr bool R_EARLY = RFX != FMT_F32 && U_EARLY && (T == 1 || KSM <= 16);      // an f32 tile is 64 registers: fetched once the up GEMV has freed them, and so are others beside too many of its own or of slices
  if (ROUTE && R_EARLY && wave < router.tiles) rraw = unit_load<RFX>(router, wave, blockIdx.x, lane);
  if (tid < T * hc) {
    float tot = ssv[0];
#pragma unroll
    for (int k = 1; k < KSM; ++k) if (k < kps) tot += ssv[k];
    const float sc = 1.0f / sqrtf(tot / (float)d + eps);
    for (int k = 0; k < kps; ++k) sls[stt * 32 + sq * kps + k] = sc;
  }
  lds_barrier(); PYRE_TS(1);
  for (int i0 = 0; i0 < n_lo; i0 += nthr) {          // (a launch-uniform count of rounds)
    const int idx = i0 + tid, t = min(hc_div(idx, rlr), T - 1);
    const float v = hc_mean(hc_slice_sum<KSM>(pv, sls + t * 32, ksplit), hc);          // slices in order, each times its stream's scale
    if (idx < n_lo) lo[idx + t * HC_PAD] = v * sigm(v);
    if (i0 + nthr < n_lo) {
      if constexpr (AHEAD) {
#pragma unroll
        for (int k = 0; k < KSM; ++k) pv[k] = pn[k];
        if (i0 + 2 * nthr < n_lo) slices(pn, idx + 2 * nthr);
      } else slices(pv, idx + nthr);
    }
  }
  if (blockIdx.x == 0 && tid < T * hc) {          // one workgroup leaves the inject rows
    float v = 0.0f;
    if (has_inject) { hc_load_slices<T, KSM>(pv, part, true, ksplit, stt, r64, lr + sq); v = hc_mean(hc_slice_sum<KSM>(pv, sls + stt * 32, ksplit), hc); }
    inj[stt * hc + sq] = v;
  }
  if constexpr (!U_EARLY) raw = unit_load<FMT>(up, s * (d >> 6) + blockIdx.x, ku, lane);
  lds_barrier(); PYRE_TS(2);
  float acc[T];
#pragma unroll
  for (int t2 = 0; t2 < T; ++t2) acc[t2] = 0.0f;
  hc_unit<FMT, T>(up, raw, ku, lane, lo + ku * 64, LP, acc);
#pragma unroll
  for (int t2 = 0; t2 < T; ++t2) red[((size_t)wave * T + t2) * 64 + lane] = acc[t2];
  if (ROUTE && !R_EARLY && wave < router.tiles) rraw = unit_load<RFX>(router, wave, blockIdx.x, lane);
  PYRE_TS(3);
  lds_barrier(); PYRE_TS(4);
  // one wave per (token, stream): the gate logit is the sum of the stream's waves in unit order; xn * sigm(gate) -> term
  for (int w = wave; w < T * hc; w += nw) {
    const int t2 = __builtin_amdgcn_readfirstlane(hc_div(w, rhc)), q = w - t2 * hc, col = blockIdx.x * 64 + lane;
    const float g = hc_unit_sum(red + ((size_t)(q * U) * T + t2) * 64 + lane, U, T * 64);
    const float xv = w == wave ? xpre : xnew[((size_t)t2 * hc + q) * d + col];
    const float nv = w == wave ? npre : norm[(size_t)q * d + col];
    term[(size_t)w * 64 + lane] = xv * sls[t2 * 32 + q * kps] * nv * sigm(g);            // rms, :209: (x * s) * w
  }
  lds_barrier();
  for (int i2 = tid; i2 < T * 64; i2 += nthr) {
    const int t2 = i2 >> 6, l = i2 & 63, col = blockIdx.x * 64 + l; float mx = 0.0f;
#pragma unroll
    for (int q = 0; q < HM; ++q) if (q < hc) mx += term[(size_t)(t2 * hc + q) * 64 + l];          // streams ascending from zero (:1380)
    const float mv = hc_mean(mx, hc);
    mixed[(size_t)t2 * d + col] = mv;
    if (ROUTE) lo[t2 * (64 + HC_PAD) + l] = mv;          // lo is free after the barrier above
  }
  PYRE_TS(5);
  if (ROUTE) {
    lds_barrier(); PYRE_TS(6);
    const size_t rr64 = (size_t)router.tiles * 64;
    for (int tile = wave; tile < router.tiles; tile += nw) {
      if (tile != wave) rraw = unit_load<RFX>(router, tile, blockIdx.x, lane);
      float ra[T];
#pragma unroll
      for (int t2 = 0; t2 < T; ++t2) ra[t2] = 0.0f;
      if constexpr (T >= PYRE_MMA_MIN) hc_unit<RFX, T>(router, rraw, blockIdx.x, lane, lo, 64 + HC_PAD, ra);
      else {
#pragma unroll 1
        for (int t2 = 0; t2 < T; ++t2) {          // one token at a time (same operations per token): T tokens at once would keep 64*T activations in registers
          float r1[1] = {0.0f};
          unit_fma<RFX, 1>(router, rraw, blockIdx.x, lds2, lane, lo + t2 * (64 + HC_PAD), 0, r1);
          rpart[((size_t)blockIdx.x * T + t2) * rr64 + (size_t)tile * 64 + lane] = r1[0];
        }
      }
      if constexpr (T >= PYRE_MMA_MIN)
#pragma unroll
        for (int t2 = 0; t2 < T; ++t2) rpart[((size_t)blockIdx.x * T + t2) * rr64 + (size_t)tile * 64 + lane] = ra[t2];
    }
  }
  PYRE_TS(7); PYRE_TS_FLUSH(hc_ts, ROUTE ? 16 : 24);
}

__global__ void k_hc_combine(float* __restrict__ x, const float* __restrict__ out, const float* __restrict__ inj, int d, int hc) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, s = blockIdx.y, ti = blockIdx.z; if (i >= d) return;
  float w = 2.0f * sigm(inj[ti * hc + s]);
  x[((size_t)ti * hc + s) * d + i] += out[(size_t)ti * d + i] * w;
}

namespace {
// Waves per workgroup and units per wave of k_hc_norm_down: a workgroup's columns must lie inside one stream, and at
// most 32 K slices fit the slice-sum buffer.
struct DownPlan { int nw, upw, ksplit; };
DownPlan down_plan(const HcDev& h) {
  int ud = h.d / 64, nw = 8; while (nw > 1 && ud % nw) nw >>= 1;
  int upw = 1; while ((h.di.U / (nw * upw)) > 32 && (ud / nw) % (2 * upw) == 0) upw *= 2;
  return DownPlan{nw, upw, h.di.U / (nw * upw)};
}

template <int FMT, int T> int norm_down_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, const DownPlan& p, const float* x_in, int in_ss, int in_ts, float* x_out,
                                               const float* comb_out, int comb_parts, const MoeOut& mo, const float* comb_inj, float eps, int nz = 1) {
  const int L = p.nw * p.upw * 64; size_t lds = 4 * ((size_t)T * (L + HC_PAD) + (size_t)p.nw * T * 64 + (size_t)p.nw * T);
  ProfScope ps(ctx, "hc_norm_down", qmat_gguf_bytes(h.di, h.di.rows) + 4.0 * T * h.hc * h.d * 4);
#define NORM_DOWN_GO(NP) hipLaunchKernelGGL((k_hc_norm_down<FMT, T, NP>), dim3(h.di.tiles, p.ksplit / h.hc, nz * h.hc), dim3(p.nw * 64), lds, ctx->stream, h.di, x_in, in_ss, in_ts, x_out, comb_out, mo, comb_inj, h.norm, h.d, h.hc, \
                     w.ssq, w.o, p.upw, (const uint2*)ctx->d_iq2xs)
  // a window's pending update as four partial vectors (pyre_hc_takes_parts); a prompt's groups of eight, whose update is summed, in an
  // instance without the gather: its instructions cost 2.7 us of 49 at 200 tokens of A3B's shape, bf16
  [[maybe_unused]] constexpr int NPT = T > 1 ? PYRE_GEMV_PARTS : 1, NPR = T == 8 ? 0 : 1;
#define NORM_DOWN_ONE(NP, FG) hipLaunchKernelGGL((k_hc_norm_down<FMT, T, NP, true, FG>), dim3(h.di.tiles, p.ksplit / h.hc, nz * h.hc), dim3(512), lds, ctx->stream, h.di, x_in, in_ss, in_ts, x_out, comb_out, mo, comb_inj, h.norm, h.d, h.hc, \
                     w.ssq, w.o, p.upw, (const uint2*)ctx->d_iq2xs)
  if constexpr (FMT == FMT_IQ3_S) { if (comb_parts > 1) NORM_DOWN_GO(PYRE_GEMV_PARTS); else NORM_DOWN_GO(1); }
  else if constexpr (FMT == FMT_BF16 || FMT == FMT_F16 || FMT == FMT_F32) {
    if (p.nw != 8 || p.upw != 1) NORM_DOWN_GO(1);
    else if (comb_parts > 1) NORM_DOWN_ONE(NPT, 0);
    // a workgroup for all row tiles prepares their columns once, one for each is the shorter chain while two of them a compute unit hold the launch
    // (five tiles, sixteen slices, us a tile each / all in one: three groups 11.3 / 17.2, four 14.3 / 17.9, six 15.0 / 17.6, eight 21.6 / 17.9, twelve 26.9 / 18.5)
    else if (T == 8 && nz > 1 && !mo.partial && (int64_t)h.di.tiles * p.ksplit * nz <= 512) NORM_DOWN_ONE(NPR, 0);
    else if (T == 8 && nz > 1 && !mo.partial) hipLaunchKernelGGL((k_hc_norm_down<FMT, T, NPR, true, 0, T == 8>), dim3(1, p.ksplit / h.hc, nz * h.hc), dim3(512), lds + 4 * (size_t)8 * T * 64, ctx->stream, h.di, x_in, in_ss, in_ts, x_out, comb_out, mo, comb_inj, h.norm, h.d, h.hc, w.ssq, w.o, p.upw, (const uint2*)ctx->d_iq2xs);          // (a workgroup prepares its columns once for all row tiles)
    else if constexpr (T == 1) { switch (mo.partial ? (mo.k + 4) / 4 : 0) { case 1: NORM_DOWN_ONE(1, 1); break; case 2: NORM_DOWN_ONE(1, 2); break; case 3: NORM_DOWN_ONE(1, 3); break; case 4: NORM_DOWN_ONE(1, 4); break; case 5: NORM_DOWN_ONE(1, 5); break; default: NORM_DOWN_ONE(1, 0); } }          // (a token's gather is the launch's longest chain)
    else NORM_DOWN_ONE(1, 0);
  }
  else NORM_DOWN_GO(1);
#undef NORM_DOWN_ONE
#undef NORM_DOWN_GO
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
template <int FMT, int T> int up_mix_rows_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, const float* xnew, float eps, float* mixed, float* inj, const HcRoute* rt, int nz) {
  const int nw = h.hc * h.up.U; size_t lds = 4 * ((size_t)T * (h.lr + HC_PAD) + (size_t)nw * T * 64 + (size_t)T * 32 + (size_t)T * h.hc * 64);
  const QMatDev rq = rt ? rt->router : QMatDev{}; float* rp = rt ? rt->part : nullptr;
  ProfScope ps(ctx, rt ? "hc_up_mix_router" : "hc_up_mix", qmat_gguf_bytes(h.up, h.up.rows) + 4.0 * T * (h.hc * h.d + h.d + (double)ksplit * (h.lr + h.hc)) +
               (rt ? qmat_gguf_bytes(rq, rq.rows) + 4.0 * T * (h.d / 64) * rq.tiles * 64 : 0.0));
#define UP_MIX_GO(...) hipLaunchKernelGGL((k_hc_up_mix<FMT, T, __VA_ARGS__>), dim3(h.d / 64, 1, nz), dim3(nw * 64), lds, ctx->stream, h.up, w.o, w.ssq, ksplit, h.di.tiles * 64, h.lr, h.hc, h.has_inject ? 1 : 0, xnew, h.norm, eps, \
                     h.d, mixed, inj, (const uint2*)ctx->d_iq2xs, rq, rp)
#define UP_MIX_R(KSM, HM) do { if (rt && rq.fmt == FMT_BF16) UP_MIX_GO(FMT_BF16, KSM, HM); else if (rt && rq.fmt == FMT_F32) UP_MIX_GO(FMT_F32, KSM, HM); else UP_MIX_GO(-1, KSM, HM); } while (0)
  // Mixes as files store them in groups of eight: the common low ranks and slice counts (widths in powers of two) have instances of their
  // own.  A launch is its instruction count -- low rank and slices at run time cost index arithmetic and a predicate a slice: A3B's
  // shape (four streams, 256, sixteen slices), 200 tokens, 58 us and with the router 82 against 39 and 60.
  constexpr bool OWN = FMT == FMT_BF16 && T == 8;
#define UP_MIX_LR(KSM) do { if (h.lr == 64) UP_MIX_F(KSM, 64); else if (h.lr == 128) UP_MIX_F(KSM, 128); else if (h.lr == 256) UP_MIX_F(KSM, 256); else UP_MIX_F(KSM, 512); } while (0)
#define UP_MIX_F(KSM, LR) do { if (rt && rq.fmt == FMT_BF16) UP_MIX_GO(FMT_BF16, KSM, 4, LR); else if (rt && rq.fmt == FMT_F32) UP_MIX_GO(FMT_F32, KSM, 4, LR); else UP_MIX_GO(-1, KSM, 4, LR); } while (0)
  bool done = false;
  if constexpr (OWN) {
    done = h.hc <= 4 && (ksplit == 8 || ksplit == 16) && (h.lr == 64 || h.lr == 128 || h.lr == 256 || h.lr == 512);
    if (done && ksplit == 16) UP_MIX_LR(16); else if (done) UP_MIX_LR(8);
  }
#undef UP_MIX_F
#undef UP_MIX_LR
  if (done) {}
  else if constexpr (FMT == FMT_BF16 || FMT == FMT_F16 || FMT == FMT_F32) { if (pyre_hc_few(h, ksplit)) UP_MIX_R(16, 4); else UP_MIX_R(32, 8); }
  else if constexpr (FMT == FMT_IQ3_S) UP_MIX_R(32, 8);
  else UP_MIX_GO(-1, 32, 8);
#undef UP_MIX_R
#undef UP_MIX_GO
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
// The formats whose products a lane forms alone; the others take sums of the activations across the wave, which then has to hold one unit.
constexpr bool up_by_columns(int fmt) { return fmt == FMT_F32 || fmt == FMT_F16 || fmt == FMT_BF16 || fmt == FMT_Q8_0 || fmt == FMT_Q4_K; }
template <int FMT, int T> int up_mix_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, const float* xnew, float eps, float* mixed, float* inj, const HcRoute* rt) {
  if constexpr (!up_by_columns(FMT)) return up_mix_rows_launch<FMT, T>(ctx, h, w, ksplit, xnew, eps, mixed, inj, rt, 1);
  else {
  const int rc = pyre_hc_up_cols_launch(ctx, h, w, ksplit, T, xnew, eps, mixed, inj); if (rc) return rc;
  return rt ? pyre_moe_router_shares_launch(ctx, "hc_up_mix_router", rt->router, mixed, T, h.d / 64, 1, rt->part, rt->dgx) : PYRE_OK;
  }
}
#define HC_T_SWITCH(F, FN, ...) \
  switch (t) { case 1: return FN<F, 1>(__VA_ARGS__); case 2: return FN<F, 2>(__VA_ARGS__); case 3: return FN<F, 3>(__VA_ARGS__); case 4: return FN<F, 4>(__VA_ARGS__); \
    case 5: return FN<F, 5>(__VA_ARGS__); case 6: return FN<F, 6>(__VA_ARGS__); case 7: return FN<F, 7>(__VA_ARGS__); default: return FN<F, 8>(__VA_ARGS__); }
#define HC_FMT_SWITCH(fmt, BODY) \
  switch (fmt) { case FMT_F32: { constexpr int F = FMT_F32; BODY } case FMT_F16: { constexpr int F = FMT_F16; BODY } case FMT_BF16: { constexpr int F = FMT_BF16; BODY } \
    case FMT_Q8_0: { constexpr int F = FMT_Q8_0; BODY } case FMT_Q4_K: { constexpr int F = FMT_Q4_K; BODY } case FMT_IQ2_XS: { constexpr int F = FMT_IQ2_XS; BODY } \
    case FMT_C4: { constexpr int F = FMT_C4; BODY } case FMT_C8: { constexpr int F = FMT_C8; BODY } \
    default: { constexpr int F = FMT_IQ3_S; BODY } }
int norm_down(pyre_ctx* ctx, const HcDev& h, const HcWork& w, const DownPlan& p, const float* x_in, int in_ss, int in_ts, float* x_out, int t, const float* comb_out, int comb_parts, const MoeOut& mo, const float* comb_inj, float eps) {
  HC_FMT_SWITCH(h.di.fmt, HC_T_SWITCH(F, norm_down_launch, ctx, h, w, p, x_in, in_ss, in_ts, x_out, comb_out, comb_parts, mo, comb_inj, eps))
}
int up_mix(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, int t, const float* xnew, float eps, float* mixed, float* inj, const HcRoute* rt) {
  HC_FMT_SWITCH(h.up.fmt, HC_T_SWITCH(F, up_mix_launch, ctx, h, w, ksplit, xnew, eps, mixed, inj, rt))
}
}  // namespace

bool pyre_hc_leaves_digits(const HcDev& h) { return pyre_hc_on_matrix_cores(h) || up_by_columns(h.up.fmt); }
bool pyre_hc_aop_ok(const HcDev& h) { return pyre_hc_on_matrix_cores(h) && h.hc <= 4; }
bool pyre_hc_takes_parts(const HcDev& h, int t) {
  const int f = h.di.fmt; const DownPlan p = down_plan(h);
  return f == FMT_IQ3_S || (t > 1 && (f == FMT_BF16 || f == FMT_F16 || f == FMT_F32) && p.nw == 8 && p.upw == 1);
}
bool pyre_hc_route_ok(const HcDev& h, const QMatDev& router) {
  const int f = h.up.fmt;
  return (f == FMT_IQ3_S || f == FMT_BF16 || f == FMT_F16 || f == FMT_F32) && (router.fmt == FMT_BF16 || router.fmt == FMT_F32) && router.cols == h.d && h.d / 64 <= 64 && router.U == h.d / 64;
}
bool pyre_hc_plan(const HcDev& h, int* nw, int* upw, int* ksplit) {
  if (h.d % 64 || h.lr % 64 || h.hc * h.up.U > 16 || h.up.tiles != h.hc * (h.d / 64) || h.di.U != h.hc * (h.d / 64)) return false;
  DownPlan p = down_plan(h); *nw = p.nw; *upw = p.upw; *ksplit = p.ksplit;
  return p.ksplit >= 1 && p.ksplit <= 32 && p.ksplit * p.nw * p.upw == h.di.U;
}
size_t pyre_hc_work_bytes(const HcDev& h) { return 256 * 4 + 2 * 4 * 8 * 32 + 4 * 8 * 32 * ((size_t)h.lr + h.hc + 64); }
void pyre_hc_work_carve(const HcDev& h, void* base, HcWork* w) {
  uint8_t* p = (uint8_t*)base; auto take = [&](size_t n) { void* r = p; p += (n + 255) & ~(size_t)255; return r; };
  w->ssq = (float*)take(4 * 8 * 32); w->smx = (float*)take(4 * 8 * 32); w->o = (float*)take(4 * 8 * 32 * ((size_t)h.lr + h.hc + 64));
}

// groups of eight tokens, the lane = row kernels (a window's launches with a group index in the grid)
static int hc_rows_split(const HcDev& h) { return down_plan(h).ksplit; }
bool pyre_hc_rows_ok(const HcDev& h) { int nw, upw, ks; return !pyre_hc_on_matrix_cores(h) && pyre_hc_plan(h, &nw, &upw, &ks); }
size_t pyre_hc_rows_bytes(const HcDev& h, int groups) { return 3 * 256 + 4 * (size_t)groups * hc_rows_split(h) * 8 * (1 + (size_t)h.di.tiles * 64); }
void pyre_hc_rows_carve(const HcDev& h, int groups, void* base, HcWork* w) { w->ssq = (float*)base; w->smx = nullptr; w->o = (float*)((uint8_t*)base + ((4 * (size_t)groups * hc_rows_split(h) * 8 + 255) & ~(size_t)255)); }
int pyre_hc_mix_rows_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, const float* x_in, int in_ss, int in_ts, float* x_out, int groups, const float* comb_out, const MoeOut* comb_moe, const float* comb_inj,
                            float eps, float* mixed, float* inj, const HcRoute* rt) {
  if (!pyre_hc_rows_ok(h) || groups < 1 || groups * h.hc > 65535 || x_in == x_out || (rt && !pyre_hc_route_ok(h, rt->router))) return pyre_fail(ctx, PYRE_E_ARG, "hc_mix_rows: unsupported shape");
  const DownPlan p = down_plan(h); const MoeOut mo = comb_moe ? *comb_moe : MoeOut{nullptr, nullptr, nullptr, 0, 0};
  int rc = [&]() -> int { HC_FMT_SWITCH(h.di.fmt, return (norm_down_launch<F, 8>(ctx, h, w, p, x_in, in_ss, in_ts, x_out, comb_out, 1, mo, comb_inj, eps, groups));) }(); if (rc) return rc;
  return [&]() -> int { HC_FMT_SWITCH(h.up.fmt, return (up_mix_rows_launch<F, 8>(ctx, h, w, p.ksplit, x_out, eps, mixed, inj, rt, groups));) }();
}

int pyre_hc_mix_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, const float* x_in, int in_ss, int in_ts, float* x_out, int t, const float* comb_out, const MoeOut* comb_moe, const float* comb_inj,
                       float eps, float* mixed, float* inj, const HcRoute* route, int comb_parts, const AopOut* aop) {
  if (t < 1 || t > 8) return pyre_fail(ctx, PYRE_E_ARG, "hc_mix: t = %d outside 1..8", t);
  if (comb_parts != 1 && !(comb_parts == PYRE_GEMV_PARTS && pyre_hc_takes_parts(h, t) && comb_out && !comb_moe)) return pyre_fail(ctx, PYRE_E_ARG, "hc_mix: %d partial vectors (1, or %d where pyre_hc_takes_parts)", comb_parts, PYRE_GEMV_PARTS);
  if (route && !pyre_hc_route_ok(h, route->router)) return pyre_fail(ctx, PYRE_E_SHAPE, "hc_mix: this router cannot ride on the mix");
  if (x_in == x_out) return pyre_fail(ctx, PYRE_E_ARG, "hc_mix: the updated streams must go to another buffer");
  if (h.d % 64 || h.lr % 64 || h.hc * h.up.U > 16 || h.up.tiles != h.hc * (h.d / 64) || h.di.U != h.hc * (h.d / 64))
    return pyre_fail(ctx, PYRE_E_SHAPE, "hc_mix: needs d and the low rank in multiples of 64 and hc * (low rank / 64) <= 16 (d %d, low rank %d, hc %d)", h.d, h.lr, h.hc);
  DownPlan p = down_plan(h);
  if (p.ksplit < 1 || p.ksplit > 32 || p.ksplit * p.nw * p.upw != h.di.U) return pyre_fail(ctx, PYRE_E_SHAPE, "hc_mix: d = %d cannot be cut into at most 32 slices of whole waves", h.d);
  const bool on_m = pyre_hc_on_matrix_cores(h);
  if (aop && !(on_m && aop->op && aop->ainv && aop->nsb >= 1 && h.hc <= 4)) return pyre_fail(ctx, PYRE_E_ARG, "hc_mix: only the matrix-core mix leaves an operand (pyre_hc_aop_ok)");
  MoeOut mo = comb_moe ? *comb_moe : MoeOut{nullptr, nullptr, nullptr, 0, 0};
  if (mo.partial && (mo.k > PYRE_MOE_KMAX || mo.d != h.d)) return pyre_fail(ctx, PYRE_E_SHAPE, "hc_mix: unreduced FFN output with top_k %d / width %d", mo.k, mo.d);
  if (on_m) {
    int rc = pyre_hc_norm_down_m_launch(ctx, h, w, x_in, in_ss, in_ts, x_out, t, comb_out, comb_parts, mo, comb_inj); if (rc) return rc;
    return pyre_hc_up_mix_m_launch(ctx, h, w, pyre_hc_m_slices(h), t, x_out, eps, mixed, inj, route, aop);
  }
  int rc = norm_down(ctx, h, w, p, x_in, in_ss, in_ts, x_out, t, comb_out, comb_parts, mo, comb_inj, eps); if (rc) return rc;
  return up_mix(ctx, h, w, p.ksplit, t, x_out, eps, mixed, inj, route);
}

int pyre_hc_combine_launch(pyre_ctx* ctx, int d, int hc, float* x, int t, const float* out, const float* inj) {
  { ProfScope ps(ctx, "hc_combine", 4.0 * t * d * (2 * hc + 1)); hipLaunchKernelGGL(k_hc_combine, dim3((d + 255) / 256, hc, t), dim3(256), 0, ctx->stream, x, out, inj, d, hc); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}
