// The second launch of a hyper-connection mix by columns: windows of a mix in a plain format, Q8_0 or Q4_K (hc.hip chooses it).
#include "hc.h"
#include <algorithm>

// The second launch of a mix (k_hc_up_mix) for a window alone, at most eight tokens, in the formats whose products a lane forms alone:
// grid (d / 16), sixteen columns a workgroup, a lane a (stream, unit, column) item of the up GEMV and TS sets of them sharing the
// tokens (set k: tokens k, k + TS, ..), on d / 16 compute units instead of d / 64; the router is a launch of its own behind it.  The
// launch is latency: fetching its code, index arithmetic, dependent reads.  Room for sixteen slices and four streams (KSM, HM)
// instead of 32 and eight is 10 KB of straight code instead of 18; bf16 mixes, what files store, have instances for low ranks of 64,
// 128, 256, 512 with exactly eight or sixteen slices (FLR > 0, widths in powers of two), which drop a predicate a slice and most
// indices.  A3B shape (four streams, 256, sixteen), bf16, one / three / eight tokens: 8.4 us a token with the larger bounds, 7.0 / 7.9 /
// 9.9 with the smaller, 5.6 / 6.4 / 7.5 with its instance (and 3.2 for router and digits; as k_hc_up_mix 8.2 a token, with the router 13.9, and
// 2.5 for the digits behind it).  A lane's terms, and every order of adding, are those of k_hc_up_mix, bit for bit.  A unit's row of lo is
// PAD floats behind the last one: the four units of a wave read four different banks.
#define PYRE_UP_PAD 68
template <int FMT, int T, int KSM, int HM, int FLR = 0> __global__ __launch_bounds__(512) void k_hc_up_mix_c(QMatDev up, const float* __restrict__ part, const float* __restrict__ ssq, int ksplit, int r64, int lr, int hc, int has_inject,
    const float* __restrict__ xnew, const float* __restrict__ norm, float eps, int d, float* __restrict__ mixed, float* __restrict__ inj) {
  constexpr int TS = T > 1 ? 2 : 1, TT = (T + TS - 1) / TS;
  const uint2* lds2 = nullptr;
  qmat_args_now(up); args_now(part, ssq, ksplit, r64, lr, hc, has_inject, xnew, norm, eps, d, mixed, inj);
  if constexpr (FLR > 0) { lr = FLR; ksplit = KSM; }
  extern __shared__ __align__(16) float sm[];
  const int nthr = blockDim.x, tid = threadIdx.x, U = lr >> 6, items = hc * U * 16;
  const float rhc = hc_recip(hc), rlr = hc_recip(lr); const int kps = __builtin_amdgcn_readfirstlane(hc_div(ksplit, rhc));
  float* lo = sm;                                          // [T][U][PAD]
  float* red = lo + (size_t)T * U * PYRE_UP_PAD;           // [hc * U][T][16]
  float* sls = red + (size_t)hc * U * T * 16;              // [T][32]: the RMS scale of the stream each slice belongs to
  const int ts = tid >= items ? (tid >= 2 * items ? 2 : 1) : 0, it = ts < TS ? tid - ts * items : 0, su = it >> 4, r = it & 15, s = hc_div(su, hc_recip(U)), ku = su - s * U, col0 = blockIdx.x * 16;
  const bool work = ts < TS;
  float ssv[KSM];
  const int stt = hc_div(tid, rhc), sq = tid - stt * hc;
  const bool own = tid < T * hc;                           // thread (token stt, stream sq): the stream's scale, and in the first workgroup its inject row
#pragma unroll
  for (int k = 0; k < KSM; ++k) ssv[k] = 0.0f;
  if (own) hc_load_run<KSM>(ssv, ssq + (size_t)(sq * kps) * T + stt, kps, T);
  // the slices of a row of lo a thread, 2 T / hc rounds (4 / hc of a single token): as many as four rounds' are fetched at once
  constexpr int NR = KSM > 16 || T == 1 ? 1 : (T == 2 ? 2 : 4);
  const int n_lo = T * lr;
  float pv[NR][KSM], pvi[KSM];
  auto slices = [&](int i0) {
#pragma unroll
    for (int r2 = 0; r2 < NR; ++r2) if (i0 + r2 * nthr < n_lo) { const int idx = i0 + r2 * nthr + tid, t = hc_div(idx, rlr); hc_load_slices<T, KSM>(pv[r2], part, idx < n_lo, ksplit, t, r64, idx - t * lr); } };
  slices(0);
  hc_load_slices<T, KSM>(pvi, part, own && has_inject && blockIdx.x == 0, ksplit, stt, r64, lr + sq);
  const UnitRaw<FMT> raw = unit_load<FMT>(up, s * (d >> 6) + (col0 >> 6), work ? ku : 0, (col0 & 63) + r);
  // the epilogue's operands: thread (token tid / 16, column tid % 16) adds the streams of its column
  float xpre[HM], npre[HM];
  const int et = tid >> 4, el = tid & 15;
#pragma unroll
  for (int q = 0; q < HM; ++q) if (tid < T * 16 && q < hc) { xpre[q] = xnew[((size_t)et * hc + q) * d + col0 + el]; npre[q] = norm[(size_t)q * d + col0 + el]; } else { xpre[q] = 0.0f; npre[q] = 0.0f; }
  if (own) {
    float tot = ssv[0];
#pragma unroll
    for (int k = 1; k < KSM; ++k) if (k < kps) tot += ssv[k];
    const float sc = 1.0f / sqrtf(tot / (float)d + eps);
    for (int k = 0; k < kps; ++k) sls[stt * 32 + sq * kps + k] = sc;
  }
  lds_barrier();
  for (int i0 = 0; i0 < n_lo; i0 += NR * nthr) {          // (a launch-uniform count of rounds)
#pragma unroll
    for (int r2 = 0; r2 < NR; ++r2) if (i0 + r2 * nthr < n_lo) {
      const int idx = i0 + r2 * nthr + tid, t = min(hc_div(idx, rlr), T - 1), i = idx - t * lr;
      const float v = hc_mean(hc_slice_sum<KSM>(pv[r2], sls + t * 32, ksplit), hc);
      if (idx < n_lo) lo[((size_t)t * U + (i >> 6)) * PYRE_UP_PAD + (i & 63)] = v * sigm(v);
    }
    if (i0 + NR * nthr < n_lo) slices(i0 + NR * nthr);
  }
  if (own && blockIdx.x == 0) inj[stt * hc + sq] = has_inject ? hc_mean(hc_slice_sum<KSM>(pvi, sls + stt * 32, ksplit), hc) : 0.0f;
  lds_barrier();
  if (work) {
    float acc[TT];
#pragma unroll
    for (int k = 0; k < TT; ++k) acc[k] = 0.0f;
    if constexpr (T % TS == 0) unit_fma<FMT, TT>(up, raw, ku, lds2, tid & 63, lo + ((size_t)ts * U + ku) * PYRE_UP_PAD, TS * U * PYRE_UP_PAD, acc);
    else {          // an odd width: the second set has a token less
      if (ts == 0) unit_fma<FMT, TT>(up, raw, ku, lds2, tid & 63, lo + ku * PYRE_UP_PAD, TS * U * PYRE_UP_PAD, acc);
      else { float a1[TT - 1]; 
#pragma unroll
        for (int k = 0; k + 1 < TT; ++k) a1[k] = 0.0f;
        unit_fma<FMT, TT - 1>(up, raw, ku, lds2, tid & 63, lo + ((size_t)ts * U + ku) * PYRE_UP_PAD, TS * U * PYRE_UP_PAD, a1);
#pragma unroll
        for (int k = 0; k + 1 < TT; ++k) acc[k] = a1[k]; }
    }
#pragma unroll
    for (int k = 0; k < TT; ++k) { const int t2 = ts + k * TS; if (t2 < T) red[((size_t)su * T + t2) * 16 + r] = acc[k]; }
  }
  lds_barrier();
  if (tid < T * 16) {
    float mx = 0.0f;
#pragma unroll
    for (int q = 0; q < HM; ++q) if (q < hc) {          // streams ascending from zero (:1380)
      const float g = hc_unit_sum(red + ((size_t)(q * U) * T + et) * 16 + el, U, T * 16);
      mx += xpre[q] * sls[et * 32 + q * kps] * npre[q] * sigm(g);            // rms, :209: (x * s) * w
    }
    mixed[(size_t)et * d + col0 + el] = hc_mean(mx, hc);
  }
}

namespace {
template <int FMT, int T> int up_cols_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, const float* xnew, float eps, float* mixed, float* inj) {
  constexpr int TS = T > 1 ? 2 : 1;
  const int items = h.hc * h.up.U * 16, nthr = std::max((TS * items + 63) / 64 * 64, (T * 16 + 63) / 64 * 64); const size_t lds = 4 * ((size_t)T * h.up.U * PYRE_UP_PAD + (size_t)items * T + (size_t)T * 32);
  ProfScope ps(ctx, "hc_up_mix", qmat_gguf_bytes(h.up, h.up.rows) + 4.0 * T * (h.hc * h.d + h.d + (double)ksplit * (h.lr + h.hc)));
#define UP_COLS_GO(...) hipLaunchKernelGGL((k_hc_up_mix_c<FMT, T, __VA_ARGS__>), dim3(h.d / 16), dim3(nthr), lds, ctx->stream, h.up, w.o, w.ssq, ksplit, h.di.tiles * 64, h.lr, h.hc, h.has_inject ? 1 : 0, xnew, h.norm, eps, h.d, mixed, inj)
  bool done = false;
  if constexpr (FMT == FMT_BF16) {
    done = h.hc <= 4 && (ksplit == 8 || ksplit == 16) && (h.lr == 64 || h.lr == 128 || h.lr == 256 || h.lr == 512);
#define UP_COLS_LR(KSM) do { if (h.lr == 64) UP_COLS_GO(KSM, 4, 64); else if (h.lr == 128) UP_COLS_GO(KSM, 4, 128); else if (h.lr == 256) UP_COLS_GO(KSM, 4, 256); else UP_COLS_GO(KSM, 4, 512); } while (0)
    if (done && ksplit == 16) UP_COLS_LR(16); else if (done) UP_COLS_LR(8);
#undef UP_COLS_LR
  }
  if (done) {}
  else if constexpr (FMT == FMT_BF16 || FMT == FMT_F16 || FMT == FMT_F32) { if (pyre_hc_few(h, ksplit)) UP_COLS_GO(16, 4); else UP_COLS_GO(32, 8); }
  else UP_COLS_GO(32, 8);
#undef UP_COLS_GO
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
template <int FMT> int up_cols(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, int t, const float* xnew, float eps, float* mixed, float* inj) {
  switch (t) { case 1: return up_cols_launch<FMT, 1>(ctx, h, w, ksplit, xnew, eps, mixed, inj); case 2: return up_cols_launch<FMT, 2>(ctx, h, w, ksplit, xnew, eps, mixed, inj);
    case 3: return up_cols_launch<FMT, 3>(ctx, h, w, ksplit, xnew, eps, mixed, inj); case 4: return up_cols_launch<FMT, 4>(ctx, h, w, ksplit, xnew, eps, mixed, inj);
    case 5: return up_cols_launch<FMT, 5>(ctx, h, w, ksplit, xnew, eps, mixed, inj); case 6: return up_cols_launch<FMT, 6>(ctx, h, w, ksplit, xnew, eps, mixed, inj);
    case 7: return up_cols_launch<FMT, 7>(ctx, h, w, ksplit, xnew, eps, mixed, inj); default: return up_cols_launch<FMT, 8>(ctx, h, w, ksplit, xnew, eps, mixed, inj); }
}
}  // namespace

int pyre_hc_up_cols_launch(pyre_ctx* ctx, const HcDev& h, const HcWork& w, int ksplit, int t, const float* xnew, float eps, float* mixed, float* inj) {
  switch (h.up.fmt) { case FMT_F32: return up_cols<FMT_F32>(ctx, h, w, ksplit, t, xnew, eps, mixed, inj); case FMT_F16: return up_cols<FMT_F16>(ctx, h, w, ksplit, t, xnew, eps, mixed, inj);
    case FMT_BF16: return up_cols<FMT_BF16>(ctx, h, w, ksplit, t, xnew, eps, mixed, inj); case FMT_Q8_0: return up_cols<FMT_Q8_0>(ctx, h, w, ksplit, t, xnew, eps, mixed, inj);
    case FMT_Q4_K: return up_cols<FMT_Q4_K>(ctx, h, w, ksplit, t, xnew, eps, mixed, inj); }
  return pyre_fail(ctx, PYRE_E_TYPE, "hc_mix: format %d has no launch by columns", h.up.fmt);
}
