// MoE FFN block: router logits -> softmax top-k (inside the gate/up launch) -> grouped expert GEMV over only the
// selected experts.
// Follows ffn / routed (f32 branch) of the reference, src/model/qwen4exp_gguf.rs:1675-1684, 1721-1732, 1754-1793,
// and top_k / soft_top / nan_clean, :3121-3139.  All experts are resident in HBM, so there is no host split.
#include "formats.h"
#include "digits.h"
#include <algorithm>
#include "gemm_m.h"
PYRE_TS_DECL(moe_ts) PYRE_TS_EXPORT(moe_ts, pyre_debug_ts_moe)

// ---- router: top-k (ties -> lower index), softmax over the chosen k in ascending expert id -----------------------------
// Runs inside every gate/up workgroup of a routed entry (all of them need the expert id before they can touch a
// weight, and a separate launch would cost more than redoing this small selection everywhere).
// Thread e sums logit e's K slices (in slice order) into shared memory.  The selection is a tournament: every wave
// of 64 logits takes its own k largest (k rounds of: the wave's largest key out of six DPP maximum steps, its lowest lane
// -- the lowest index -- from a ballot, that lane retires its key), the waves' candidates meet in shared memory, each
// candidate counts the candidates that beat it (larger key, or equal key and lower index) and the k that are beaten by
// fewer than k others are the choice.  Leaves the chosen ids (ascending) in s_idx[0..k) and their logits in s_val[0..k).
struct RouteLds { float lv[1024]; float r_val[32]; float s_val[32]; int s_idx[32]; float s_w[32]; uint64_t cand[512 + 96]; uint64_t win[32]; };          // (cand: read in runs of 96)
#ifdef PYRE_PHASE_TS
#define ROUTE_TS_PARAM , unsigned long long* rts_
#define ROUTE_TS_ARG , ts_
#define ROUTE_TS(k) rts_[k] = wall_clock64()
#else
#define ROUTE_TS_PARAM
#define ROUTE_TS_ARG
#define ROUTE_TS(k)
#endif
// A logit becomes a 32-bit key whose unsigned order is the logits' order (0 = no candidate).
__device__ __forceinline__ uint32_t route_key(float v) {
  uint32_t u = __float_as_uint(v + 0.0f);          // -0 counts as +0, as in a float comparison
  return u ^ ((u & 0x80000000u) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float route_key_value(uint32_t u) { return __uint_as_float(u ^ ((u & 0x80000000u) ? 0x80000000u : 0xFFFFFFFFu)); }
template <int CTRL> __device__ __forceinline__ uint32_t route_dpp(uint32_t m) {          // lanes without a source see 0, the maximum's identity: the move folds into the v_max
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, CTRL, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t route_wave_max(uint32_t m) {          // idempotent, so the row broadcasts need no row masks
  m = max(m, route_dpp<0x111>(m)); m = max(m, route_dpp<0x112>(m)); m = max(m, route_dpp<0x114>(m)); m = max(m, route_dpp<0x118>(m));      // row_shr 1, 2, 4, 8: lane 15 of a row holds the row's
  m = max(m, route_dpp<0x142>(m)); m = max(m, route_dpp<0x143>(m));          // row_bcast 15, 31: lane 63 holds the wave's
  return (uint32_t)__builtin_amdgcn_readlane((int)m, 63);
}
// called by the whole workgroup of NT threads (at least n_exp, a multiple of 64), after lv[] is complete
template <int NT>
__device__ __forceinline__ void route_select(int n_exp, int k, RouteLds& L) {
  const int e = threadIdx.x, lane = e & 63, wave = e >> 6, nwv = (n_exp + 63) >> 6;
  if (wave < nwv) {
    uint32_t key = e < n_exp ? route_key(L.lv[e]) : 0u;
    uint32_t ck = 0u, cl = 0u;          // lane r keeps the wave's r-th candidate
    for (int round = 0; round < k; ++round) {
      const uint32_t wm = route_wave_max(key);
      const int ol = __builtin_ctzll((unsigned long long)__ballot(key == wm));          // the lowest lane that holds it = the lowest index
      ck = lane == round ? wm : ck; cl = lane == round ? (uint32_t)ol : cl;
      key = lane == ol ? 0u : key;
    }
    if (lane < k) L.cand[wave * k + lane] = ((uint64_t)ck << 32) | (uint32_t)(0xFFFFFFFFu - ((uint32_t)(wave * 64) + cl));
  }
  lds_barrier();
  // eight neighbouring lanes share a candidate and split the others among them; larger 64-bit word = larger key, or the
  // same key at a lower index: a strict order, so the k winners hold the ranks 0 .. k-1
  const int nc = nwv * k, sub = e & 7;
  for (int i = e >> 3; i < nc; i += NT / 8) {
    const uint64_t ci = L.cand[i];
    int beaten = 0;
    for (int jb = 0; jb < nc; jb += 96) {          // (twelve reads in flight before the first comparison: one round for eight waves' twelve candidates)
      uint64_t cj[12];
#pragma unroll
      for (int r = 0; r < 12; ++r) cj[r] = L.cand[jb + sub + 8 * r];
#pragma unroll
      for (int r = 0; r < 12; ++r) beaten += (jb + sub + 8 * r < nc && cj[r] > ci) ? 1 : 0;
    }
    beaten += __builtin_amdgcn_mov_dpp(beaten, 0xB1, 0xf, 0xf, true);          // quad_perm [1,0,3,2]
    beaten += __builtin_amdgcn_mov_dpp(beaten, 0x4E, 0xf, 0xf, true);          // quad_perm [2,3,0,1]
    beaten += __builtin_amdgcn_mov_dpp(beaten, 0x141, 0xf, 0xf, true);         // row_half_mirror: the other quad of the eight
    if (sub == 0 && (uint32_t)(ci >> 32) != 0u && beaten < k) L.win[beaten] = ci;
  }
  lds_barrier();
  if (wave == 0) {
    const uint64_t w = L.win[min(lane, 31)];
    const uint32_t idx = 0xFFFFFFFFu - (uint32_t)w;
    int pos = 0;
    for (int j = 0; j < k; ++j) { const uint32_t oj = (uint32_t)__builtin_amdgcn_readlane((int)idx, j); pos += oj < idx ? 1 : 0; }
    if (lane < k) { L.s_idx[pos] = (int)idx; L.s_val[pos] = route_key_value((uint32_t)(w >> 32)); }
  }
}
// The logits are given as nsl (<= 64) K-slice sums `sstride` floats apart, added in slice order (nsl == 1: the logits
// themselves); all slices are fetched before the first add, in groups of eight behind launch-uniform branches.  NT: the threads of the
// workgroup; NSM: a bound of nsl.
template <int NT, int NSM = 64>
__device__ __forceinline__ void route_topk(const float* __restrict__ logits, int nsl, int sstride, int n_exp, int k, RouteLds& L ROUTE_TS_PARAM) {
  const int e = threadIdx.x;
  if constexpr (NSM == 1) { if (e < n_exp) { const float v = logits[e]; L.lv[e] = isnan(v) ? -INFINITY : v; } }
  else if (e < n_exp) {
    float sv[NSM];
#pragma unroll
    for (int q = 0; q < NSM; ++q) sv[q] = 0.0f;
#pragma unroll
    for (int g = 0; g < NSM / 8; ++g) if (g * 8 < nsl) {
#pragma unroll
      for (int q = 0; q < 8; ++q) sv[g * 8 + q] = (logits + (size_t)min(g * 8 + q, nsl - 1) * sstride)[e];
    }
    float v = sv[0];
#pragma unroll
    for (int g = 0; g < NSM / 8; ++g) {
      if (g * 8 + 8 <= nsl) {          // (a whole group carries no predicates)
#pragma unroll
        for (int q = g ? 0 : 1; q < 8; ++q) v += sv[g * 8 + q];
      } else {
#pragma unroll
        for (int q = g ? 0 : 1; q < 8; ++q) if (g * 8 + q < nsl) v += sv[g * 8 + q];
      }
    }
    if (isnan(v)) v = -INFINITY;      // nan_clean
    L.lv[e] = v;
  }
  ROUTE_TS(5);
  lds_barrier(); ROUTE_TS(6);
  route_select<NT>(n_exp, k, L);
  ROUTE_TS(7);
  lds_barrier();
}
// softmax over the chosen logits in ascending expert id (soft_top); called by the whole workgroup after route_topk
__device__ __forceinline__ void route_weights(int k, RouteLds& L) {
  const int e = threadIdx.x;
  float mx = -INFINITY, ex = 1.0f;
  // the k (<= 32) values in order, eight in flight at a time
  auto walk = [&](const float (&p)[32], auto&& f) {
#pragma unroll
    for (int g = 0; g < 32; g += 8) if (g < k) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = p[g + i];
#pragma unroll
      for (int i = 0; i < 8; ++i) if (g + i < k) f(v[i]);
    } };
  if (e < k) { walk(L.s_val, [&](float v) { mx = fmaxf(mx, v); }); ex = isfinite(mx) ? expf(L.s_val[e] - mx) : 1.0f; L.r_val[e] = ex; }
  lds_barrier();
  if (e < k) {
    float w;
    if (!isfinite(mx)) w = 1.0f / (float)k;
    else { float sum = 0.0f; walk(L.r_val, [&](float v) { sum += v; }); w = ex / sum; }
    L.s_w[e] = w;
  }
}

// ---- routing + expert gate/up: h[entry][r] = silu(gate[r] . x) * (up[r] . x) -------------------------------------------
// grid (row tiles, entries), 16 waves; entry = ti*(k+1) + j, j < k: the j-th chosen expert of token ti (ascending id),
// j == k: the shared expert.  Tile 0 of entry (ti, 0) publishes the token's expert ids and weights, tile 0 of the shared
// entry publishes the shared-expert gate sigmoid(sh_gate_inp . x).
// The K range is cut into P parts of NW wave shares each; a dot product is the sum of its parts in order from the
// first, a part the sum of its wave shares in wave order -- whatever the launch shape, so a token's result does not
// depend on it.  gridDim.z == 1: the workgroup's wave w takes share w of every part (P accumulators) and stores
// silu(g) * u.  gridDim.z == nz > 1 (P == 1 in the template, nz parts): workgroup kz takes part kz only -- an entry's 64
// rows on nz compute units instead of one; at one token a launch of tiles x (k+1) workgroups leaves most of the chip
// idle -- and leaves the part's raw sums, gate at h[((entry*nz + kz)*2 + 0)*hstride + row], up at [... + 1]; the down
// launch adds the parts and forms silu(g) * u with the same operations.
// The window form (PRE, both parts in the workgroup) is held to 64 registers for the formats whose decode fits them
// (next to) without spilling, so that two workgroups share a compute unit: five tokens' 440 workgroups are then resident
// at once instead of taking a second turn on the 256 compute units.
// PRE: the token's experts were chosen by k_moe_route (windows of several tokens: hundreds of workgroups would each redo
// the selection otherwise); the workgroup reads its expert id and publishes nothing but the shared-expert gate.
// FIX: the A3B configuration's constants (512 experts, top 10, d = 2048 in 32 router slices, ff = 512) folded in at compile
// time (the launcher checks them) -- same arithmetic.
// ID (IQ3_S): the dot products in the integer form of digits.h -- 1.4 vector instructions a weight where byte -> float and
// multiply-add take 3; dgx holds the digits of the window's activations, token ti at dgx + ti * (d / 64) * DGX_STRIDE.
// perm (a launch for hundreds of tokens): workgroup y takes entry perm[y], the routed entries by expert, so that an expert's
// weights are in the second-level caches for all of its tokens; the shared expert's entries follow
__device__ __forceinline__ int entry_of(const int32_t* __restrict__ perm, int y, int T, int top_k) { return __builtin_amdgcn_readfirstlane(y < T * top_k ? perm[y] : (y - T * top_k) * (top_k + 1) + top_k); }
template <int FMT, int NW, int P, bool PRE, bool FIX = false, bool ID = false>
__global__ __launch_bounds__(NW * 64, (PRE && P == 2 && FMT >= 5 && FMT <= 7) ? 8 : 1) void k_moe_gu(MoeDev m, const float* __restrict__ logits, int32_t* __restrict__ sel_idx, float* __restrict__ sel_w, float* __restrict__ sg,
                                                   const float* __restrict__ x, float* __restrict__ h, int hstride, const uint2* __restrict__ g2, int nsl, int sstride, int tstride, const uint32_t* __restrict__ dgx,
                                                   uint32_t* __restrict__ dgh, const int32_t* __restrict__ perm) {
  static_assert(!ID || FMT == FMT_IQ3_S, "the integer form is IQ3_S's");
  const uint2* lds2 = nullptr;          // no format needs a codebook in shared memory any more
  PYRE_TS_VARS PYRE_TS(0);
  args_now(m.n_exp, m.top_k, logits, nsl, sstride, tstride);          // what the selection needs; the rest would crowd the scalar registers the activations go through
  const int n_exp = FIX ? 512 : m.n_exp, top_k = FIX ? 10 : m.top_k, d = FIX ? 2048 : m.d, ff = FIX ? 512 : m.ff;
  if constexpr (FIX) nsl = 32;
  __shared__ float red[2][P][NW][64];
  __shared__ RouteLds rl;
  __shared__ uint8_t hsm[ID ? 3 : 1][64];
  const int k1 = top_k + 1; int entry = blockIdx.y;
  if constexpr (PRE) if (perm) entry = entry_of(perm, entry, (int)gridDim.y / k1, top_k);
  const int ti = entry / k1, j = entry % k1;
  const bool shared = j == top_k;
  const int nrows = shared ? m.sf : ff;
  if ((int)blockIdx.x * 64 >= nrows) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const float* xs = x + (size_t)ti * d;
  int expert = 0;
  if (!shared) {
    if constexpr (PRE) expert = __builtin_amdgcn_readfirstlane(sel_idx[ti * top_k + j]);
    else { route_topk<NW * 64>(logits + (size_t)ti * tstride, nsl, sstride, n_exp, top_k, rl ROUTE_TS_ARG); expert = __builtin_amdgcn_readfirstlane(rl.s_idx[j]); }
  } else if (blockIdx.x == 0) {
    float p = 0.0f;
    for (int ib = threadIdx.x; ib < d; ib += 4 * NW * 64) {          // four elements per pass, loads first (elements past d: weight zero)
      float a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) { const int ic = min(ib + u * NW * 64, d - 1); a[u] = m.sh_gate_inp[ic]; b[u] = xs[ic]; }
#pragma unroll
      for (int u = 0; u < 4; ++u) if (ib + u * NW * 64 < d) p = fmaf(a[u], b[u], p);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) p += __shfl_xor(p, o);
    if (lane == 0) red[0][0][wave][0] = p;
    lds_barrier();
    if (threadIdx.x == 0) { float tot = 0.0f; for (int w = 0; w < NW; ++w) tot += red[0][0][w][0]; rl.s_w[0] = 1.0f / (1.0f + expf(-tot)); }
    lds_barrier();
  }
  PYRE_TS(1);
  const QMatDev& G = shared ? m.sh_gate : m.gate_e; const QMatDev& Up = shared ? m.sh_up : m.up_e;
  const int tile = (shared ? 0 : expert * (ff >> 6)) + blockIdx.x;
  const int nz = (FIX && !PRE) ? 2 : (FIX ? 1 : (int)gridDim.z), kz = blockIdx.z, np = P * nz;          // np parts in all (FIX: two workgroups a single token's entry, one a window's)
  const int GU = FIX ? 32 : G.U;          // 64-column units of a row (both matrices, routed or shared: d / 64)
  const int upw = (GU + NW * np - 1) / (NW * np);
  const uint32_t* dgs = ID ? dgx + (size_t)ti * GU * DGX_STRIDE : nullptr;
  // one unit of a matrix into an accumulator, in the f32 or the integer form
  auto mac = [&](const QMatDev& Q, const UnitRaw<FMT>& r, int ku, float (&a)[1]) {
    if constexpr (ID) unit_idot_iq3s(r, dgs + (size_t)ku * DGX_STRIDE, a[0]);
    else unit_fma<FMT, 1>(Q, r, ku, lds2, lane, xs + ku * 64, 0, a);
  };
  float ag[P][1], au[P][1];
#pragma unroll
  for (int p = 0; p < P; ++p) { ag[p][0] = 0.0f; au[p][0] = 0.0f; }
  if (P == 2 && upw == 1) {
    // one unit per part: both parts' units of both matrices are fetched before the first is consumed
    const int ka = min(2 * wave, GU - 1), kb = min(2 * wave + 1, GU - 1);
    UnitRaw<FMT> g0 = unit_load<FMT>(G, tile, ka, lane), u0 = unit_load<FMT>(Up, tile, ka, lane), g1 = unit_load<FMT>(G, tile, kb, lane), u1 = unit_load<FMT>(Up, tile, kb, lane);
    if (2 * wave < GU) { mac(G, g0, ka, ag[0]); mac(Up, u0, ka, au[0]); }
    if (2 * wave + 1 < GU) { mac(G, g1, kb, ag[P - 1]); mac(Up, u1, kb, au[P - 1]); }
  } else {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int k0 = min(GU, (wave * np + kz * P + p) * upw), kend = min(GU, k0 + upw);          // wave w's shares of the np parts are adjacent
      // two units of both matrices are fetched before the first is consumed: a rolled loop would pay a memory round trip per unit
      for (int ku = k0; ku < kend; ku += 2) {
        const int kb = min(ku + 1, kend - 1);
        UnitRaw<FMT> g0 = unit_load<FMT>(G, tile, ku, lane), u0 = unit_load<FMT>(Up, tile, ku, lane), g1 = unit_load<FMT>(G, tile, kb, lane), u1 = unit_load<FMT>(Up, tile, kb, lane);
        mac(G, g0, ku, ag[p]); mac(Up, u0, ku, au[p]);
        if (ku + 1 < kend) { mac(G, g1, ku + 1, ag[p]); mac(Up, u1, ku + 1, au[p]); }
      }
    }
  }
#pragma unroll
  for (int p = 0; p < P; ++p) { red[0][p][wave][lane] = ag[p][0]; red[1][p][wave][lane] = au[p][0]; }
  PYRE_TS(2);
  lds_barrier(); PYRE_TS(3);
  if (threadIdx.x < 64) {
    float g = 0.0f, u = 0.0f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      float gp = red[0][p][0][lane], up = red[1][p][0][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) { gp += red[0][p][w][lane]; up += red[1][p][w][lane]; }
      if (p == 0) { g = gp; u = up; } else { g += gp; u += up; }
    }
    if (nz == 1) {
      float s = 1.0f / (1.0f + expf(-g));
      const float hv = (g * s) * u;      // silu(g) * u, silu(x) = x * sigm(x)
      h[(size_t)entry * hstride + blockIdx.x * 64 + lane] = hv;
      // the tile's 64 rows are one unit of the down product's columns: their digits for its integer form
      if constexpr (ID) { if (dgh) digits_eo_wave(hv, lane, hsm, dgh + ((size_t)entry * (hstride >> 6) + blockIdx.x) * DGX_STRIDE); }
    } else {
      float* hp = h + ((size_t)entry * nz + kz) * 2 * hstride + blockIdx.x * 64 + lane;
      hp[0] = g; hp[hstride] = u;
    }
  }
  // Publishing comes last: a global store ahead of the dot products would stop the compiler from keeping the
  // activations in scalar registers (it could no longer prove them unmodified).
  if (blockIdx.x == 0 && kz == 0) {
    if (shared) { if (threadIdx.x == 0) sg[ti] = rl.s_w[0]; }
    else if (!PRE && j == 0) {
      route_weights(top_k, rl);       // thread e < k writes and then reads its own s_w entry
      if ((int)threadIdx.x < top_k) { sel_idx[ti * top_k + threadIdx.x] = rl.s_idx[threadIdx.x]; sel_w[ti * top_k + threadIdx.x] = rl.s_w[threadIdx.x]; }
    }
  }
  PYRE_TS(4); PYRE_TS_FLUSH(moe_ts, 0);
}

// ---- routing alone (windows of several tokens): grid t, 1024 threads; ids ascending and softmax weights of token ti ------
// K > 0: the experts a token (m.top_k) at compile time: the selection's loops are a chain of some forty steps a count (512 experts, top
// 10, sixteen slices: 4.5 us with the count at run time, 3.8 with it folded).  NSM: a bound of the router slices, whose sums' registers
// and predicates the compiler lays out for it.
template <int K, int NSM>
__global__ __launch_bounds__(1024) void k_moe_route(MoeDev m, const float* __restrict__ logits, int32_t* __restrict__ sel_idx, float* __restrict__ sel_w, int nsl, int sstride, int tstride) {
  __shared__ RouteLds rl;
  const int ti = blockIdx.x, n_exp = m.n_exp, top_k = K ? K : m.top_k;
  args_now(n_exp, top_k, logits, sel_idx, sel_w, nsl, sstride, tstride);
#ifdef PYRE_PHASE_TS
  unsigned long long ts_[8];
#endif
  route_topk<1024, NSM>(logits + (size_t)ti * tstride, nsl, sstride, n_exp, top_k, rl ROUTE_TS_ARG);
  route_weights(top_k, rl);
  if ((int)threadIdx.x < top_k) { sel_idx[ti * top_k + threadIdx.x] = rl.s_idx[threadIdx.x]; sel_w[ti * top_k + threadIdx.x] = rl.s_w[threadIdx.x]; }
}

// ---- expert down: partial[entry][r] = down[r] . h[entry] ---------------------------------------------------------------
// NZ > 1: h arrives as the gate / up sums of NZ K parts (k_moe_gu with gridDim.z = NZ); each wave forms the 64 values of
// a unit, silu(sum of gate parts) * (sum of up parts), in its own slice of shared memory while the unit's weights are
// on their way (a wave's shared-memory operations execute in order: no workgroup barrier).
// ID (IQ3_S): the integer form of digits.h on the digits of h -- left by k_moe_gu beside h (NZ == 1), or formed here by
// the wave that forms the unit's values (NZ > 1); the same digits either way, so a token's bits do not depend on the form.
template <int FMT, int NW, int NZ, bool FIX = false, bool ID = false>
__global__ __launch_bounds__(NW * 64) void k_moe_down(MoeDev m, const int32_t* __restrict__ sel_idx, const float* __restrict__ h, int hstride, float* __restrict__ partial,
                                                     const uint2* __restrict__ g2, const uint32_t* __restrict__ dgh, const int32_t* __restrict__ perm) {
  static_assert(!ID || FMT == FMT_IQ3_S, "the integer form is IQ3_S's");
  const uint2* lds2 = nullptr;          // no format needs a codebook in shared memory any more
  PYRE_TS_VARS PYRE_TS(0);
  qmat_args_now(m.down_e); qmat_args_now(m.sh_down); args_now(m.d, m.top_k, sel_idx, h, hstride, partial);
  const int top_k = FIX ? 10 : m.top_k, d = FIX ? 2048 : m.d;          // FIX: the A3B configuration (top 10, d = 2048, routed and shared experts 512 wide), checked by the launcher
  __shared__ float red[NW][64];
  __shared__ float hx[(NZ > 1 && !ID) ? NW : 1][64];
  __shared__ __align__(16) uint32_t hdg[(NZ > 1 && ID) ? NW : 1][DGX_STRIDE];
  __shared__ uint8_t hsm[(NZ > 1 && ID) ? NW : 1][3][64];
  const int k1 = top_k + 1; int entry = blockIdx.y;
  if constexpr (NZ == 1) if (perm) entry = entry_of(perm, entry, (int)gridDim.y / k1, top_k);
  const int ti = entry / k1, j = entry % k1;
  const bool shared = j == top_k;
  const QMatDev& D = shared ? m.sh_down : m.down_e;
  const int tile = (shared ? 0 : sel_idx[ti * top_k + j] * (d >> 6)) + blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int DU = FIX ? 8 : D.U;
  const int upw = (DU + NW - 1) / NW, k0 = wave * upw, kend = min(DU, k0 + upw);
  float acc[1] = {0.0f};
  if constexpr (NZ == 1) {
    const float* xs = h + (size_t)entry * hstride;
    if constexpr (ID) {
      const uint32_t* dge = dgh + (size_t)entry * (hstride >> 6) * DGX_STRIDE;
      for (int ku = k0; ku < kend; ++ku) { UnitRaw<FMT> r = unit_load<FMT>(D, tile, ku, lane); unit_idot_iq3s(r, dge + (size_t)ku * DGX_STRIDE, acc[0]); }
    } else
    for (int ku = k0; ku < kend; ++ku) unit_dot<FMT, 1>(D, lds2, tile, ku, lane, xs + ku * 64, 0, acc);
  } else {
    const float* hp = h + (size_t)entry * NZ * 2 * hstride + lane;
    for (int ku = k0; ku < kend; ++ku) {
      UnitRaw<FMT> r = unit_load<FMT>(D, tile, ku, lane);
      float gp[NZ], up[NZ];
#pragma unroll
      for (int q = 0; q < NZ; ++q) { gp[q] = hp[(size_t)(2 * q) * hstride + ku * 64]; up[q] = hp[(size_t)(2 * q + 1) * hstride + ku * 64]; }
      float g = gp[0], u = up[0];
#pragma unroll
      for (int q = 1; q < NZ; ++q) { g += gp[q]; u += up[q]; }
      float s = 1.0f / (1.0f + expf(-g));
      __builtin_amdgcn_wave_barrier();
      if constexpr (ID) {
        digits_eo_wave((g * s) * u, lane, hsm[wave], hdg[wave]);
        __builtin_amdgcn_wave_barrier();
        unit_idot_iq3s(r, hdg[wave], acc[0]);
      } else {
        hx[wave][lane] = (g * s) * u;
        __builtin_amdgcn_wave_barrier();
        unit_fma<FMT, 1>(D, r, ku, lds2, lane, hx[wave], 0, acc);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  red[wave][lane] = acc[0];
  PYRE_TS(1);
  lds_barrier(); PYRE_TS(2);
  if (threadIdx.x < 64) {
    float s = red[0][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[w][lane];
    partial[(size_t)entry * d + blockIdx.x * 64 + lane] = s;
  }
  PYRE_TS(3); PYRE_TS_FLUSH(moe_ts, 8);
}

// y[ti][r]: the four group sums of moe_out_value, added in order (few experts only: top_k <= PYRE_MOE_KMAX; more experts
// take the plain sum shared * sg + (the experts' terms in ascending id, from zero))
__global__ void k_moe_sum(const float* __restrict__ partial, const float* __restrict__ sel_w, const float* __restrict__ sg, int d, int k, float* __restrict__ y) {
  int r = blockIdx.x * blockDim.x + threadIdx.x, ti = blockIdx.y; if (r >= d) return;
  if (k <= PYRE_MOE_KMAX) { const MoeOut mo{partial, sel_w, sg, d, k}; y[(size_t)ti * d + r] = moe_out_value(mo, ti, r); return; }
  const float* p = partial + (size_t)ti * (k + 1) * d;
  float o = 0.0f; for (int j = 0; j < k; ++j) o += sel_w[ti * k + j] * p[(size_t)j * d + r];
  float yv = p[(size_t)k * d + r] * sg[ti];
  y[(size_t)ti * d + r] = yv + o;
}

// ---- expert down of a window, summed by groups: parts[(q*t + ti)*d + r] = P_q of moe_out_value -------------------------------
// grid (d/64, t, PYRE_MOE_GROUPS), NW waves.  The workgroup computes the down rows of its group's (at most PYRE_MOE_GMAX)
// entries as k_moe_down does -- wave w the K share w of every entry, the shares added in wave order -- and folds them with
// the routing weights in the group's order: the consumer then reads four vectors a token instead of k + 1, and the value is
// bit for bit what moe_out_value forms from k_moe_down's unreduced terms.  A wave's weights of all entries and its slices
// of their activations (through its own shared memory: no workgroup barrier) are fetched before the first is used.
// GE: entries a group can hold in this instance (3 covers top_k <= 11, PYRE_MOE_GMAX the rest) -- the register budget follows it.
// ID (IQ3_S): the integer form on the digits k_moe_gu left beside h, as k_moe_down<.., ID>.
template <int FMT, int NW, int GE, bool FIX = false, bool ID = false>
__global__ __launch_bounds__(NW * 64, (GE <= 3 && FMT >= 5 && FMT <= 7) ? 6 : 1) void k_moe_down_groups(MoeDev m, const int32_t* __restrict__ sel_idx, const float* __restrict__ sel_w, const float* __restrict__ sg,
                                                            const float* __restrict__ h, int hstride, float* __restrict__ parts, const uint2* __restrict__ g2, const uint32_t* __restrict__ dgh) {
  static_assert(GE <= PYRE_MOE_GMAX, "a group holds at most PYRE_MOE_GMAX entries");
  static_assert(!ID || FMT == FMT_IQ3_S, "the integer form is IQ3_S's");
  const uint2* lds2 = nullptr;
  qmat_args_now(m.down_e); qmat_args_now(m.sh_down); args_now(m.d, m.top_k, sel_idx, h, hstride, parts);
  __shared__ float red[GE][NW][64];
  __shared__ float hx[ID ? 1 : NW][GE][64];
  __shared__ __align__(16) uint32_t hdg[ID ? NW : 1][GE][DGX_STRIDE];
  const int ti = blockIdx.y, q = blockIdx.z, k = FIX ? 10 : m.top_k, gsz = (k + 4) / 4, d = FIX ? 2048 : m.d;          // FIX: the A3B configuration (top 10, d = 2048, experts 512 wide), checked by the launcher
  const int j0 = min(k, q * gsz), nr = min(k, j0 + gsz) - j0;          // the group's routed entries j0 .. j0+nr-1
  const bool with_shared = q == PYRE_MOE_GROUPS - 1;
  const int ne = nr + (with_shared ? 1 : 0);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // the routed and the shared matrices may differ in width: each has its own K shares (as in k_moe_down)
  const int Ur = FIX ? 8 : m.down_e.U, Us = FIX ? 8 : m.sh_down.U, upr = (Ur + NW - 1) / NW, ups = (Us + NW - 1) / NW;
  const int niter = max(nr > 0 ? upr : 0, with_shared ? ups : 0);
  int tile[GE]; const float* xs[GE]; const uint32_t* dge[GE];
#pragma unroll
  for (int e = 0; e < GE; ++e) {
    const bool shared = with_shared && e == nr; const int j = shared ? k : min(j0 + e, k - 1);
    tile[e] = (shared ? 0 : __builtin_amdgcn_readfirstlane(sel_idx[ti * k + j]) * (d >> 6)) + blockIdx.x;
    xs[e] = h + (size_t)(ti * (k + 1) + j) * hstride;
    dge[e] = ID ? dgh + (size_t)(ti * (k + 1) + j) * (hstride >> 6) * DGX_STRIDE : nullptr;
  }
  float acc[GE][1];
#pragma unroll
  for (int e = 0; e < GE; ++e) acc[e][0] = 0.0f;
  // the routing weights and the shared expert's gate are requested now, not behind the products
  float wv[GE];
#pragma unroll
  for (int e = 0; e < GE; ++e) wv[e] = e < nr ? sel_w[ti * k + j0 + e] : 0.0f;
  const float g = with_shared ? sg[ti] : 0.0f;
  for (int it = 0; it < niter; ++it) {
    UnitRaw<FMT> r[GE]; float hv[GE]; bool on[GE]; int ku[GE];
#pragma unroll
    for (int e = 0; e < GE; ++e) {
      const bool shared = with_shared && e == nr; const int up = shared ? ups : upr, U = shared ? Us : Ur;
      ku[e] = wave * up + it; on[e] = e < ne && it < up && ku[e] < U;
      if (on[e]) { const QMatDev& D = shared ? m.sh_down : m.down_e; r[e] = unit_load<FMT>(D, tile[e], ku[e], lane); if constexpr (!ID) hv[e] = xs[e][ku[e] * 64 + lane]; }
    }
    if constexpr (ID) {
      // the units' digits through the wave's own shared memory: one coalesced load an entry, all in flight with the weights
      // (as scalar loads they would come one entry after the other: three entries' digits do not fit the scalar registers)
      uint32_t dv[GE];
#pragma unroll
      for (int e = 0; e < GE; ++e) dv[e] = on[e] ? (dge[e] + (size_t)ku[e] * DGX_STRIDE)[lane] : 0u;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int e = 0; e < GE; ++e) if (on[e]) hdg[wave][e][lane] = dv[e];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int e = 0; e < GE; ++e) if (on[e]) unit_idot_iq3s(r[e], hdg[wave][e], acc[e][0]);
      __builtin_amdgcn_wave_barrier();
    } else {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int e = 0; e < GE; ++e) if (on[e]) hx[wave][e][lane] = hv[e];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int e = 0; e < GE; ++e) if (on[e]) { const QMatDev& D = (with_shared && e == nr) ? m.sh_down : m.down_e; unit_fma<FMT, 1>(D, r[e], ku[e], lds2, lane, hx[wave][e], 0, acc[e]); }
      __builtin_amdgcn_wave_barrier();
    }
  }
#pragma unroll
  for (int e = 0; e < GE; ++e) if (e < ne) red[e][wave][lane] = acc[e][0];
  lds_barrier();
  if (threadIdx.x < 64) {
    float o = 0.0f;
#pragma unroll
    for (int e = 0; e < GE; ++e) if (e < ne) {
      float pv = red[e][0][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) pv += red[e][w][lane];
      if (e < nr) o = fmaf(wv[e], pv, o); else o = fmaf(pv, g, o);          // the shared expert comes last
    }
    parts[((size_t)q * gridDim.y + ti) * d + blockIdx.x * 64 + lane] = o;
  }
}

// the digits of t tokens' activations as a launch of its own (callers whose producer kernel does not leave them): grid (d / 64, t), one wave
__global__ __launch_bounds__(64) void k_act_digits_eo(const float* __restrict__ x, int d, uint32_t* __restrict__ dgx) {
  __shared__ uint8_t sm[3][64];
  const int ku = blockIdx.x, ti = blockIdx.y, lane = threadIdx.x;
  digits_eo_wave(x[(size_t)ti * d + ku * 64 + lane], lane, sm, dgx + ((size_t)ti * (d >> 6) + ku) * DGX_STRIDE);
}

// The router's product by the shares of its GEMV's waves, and (further workgroups, one wave each) the digits of the activations: grid
// tiles * nw + (d / 64) * t, one wave.  Share w of row tile b: units [w * upw, + upw) of every token, part[(w * t + ti) * tiles * 64 + row].
// A share is what wave w of k_gemv forms; added in wave order they are its sum, bit for bit.  NG = 0: a single token, its activations as scalar
// loads; else NG groups of four tokens at once (unit_mma): a token after the other each waited for its own scalar loads and for the weights
// again (A3B's router, one token 2.8 us; four 6.7 -> 3.7, eight 4.0; the block of four tokens 31.8 -> 29.5, of eight 44.4 -> 38.3).
template <int RF, int NG>
__global__ __launch_bounds__(64) void k_moe_router_shares(QMatDev q, const float* __restrict__ x, int t, int d, int nw, int upw, float* __restrict__ part, uint32_t* __restrict__ dgx) {
  __shared__ uint8_t sm[3][64];
  const int lane = threadIdx.x, ns = q.tiles * nw, b = blockIdx.x;
  if (b >= ns) { const int ku = (b - ns) % (d >> 6), ti = (b - ns) / (d >> 6); digits_eo_wave(x[(size_t)ti * d + ku * 64 + lane], lane, sm, dgx + ((size_t)ti * (d >> 6) + ku) * DGX_STRIDE); return; }
  const int tile = b / nw, w = b - tile * nw, k0 = w * upw, k1 = min((int)q.U, k0 + upw);
  const size_t r64 = (size_t)q.tiles * 64;
  if constexpr (NG == 0) {
    const uint2* lds2 = nullptr; float acc[1] = {0.0f};
    for (int ku = k0; ku < k1; ++ku) { const UnitRaw<RF> r = unit_load<RF>(q, tile, ku, lane); unit_fma<RF, 1>(q, r, ku, lds2, lane, x + ku * 64, 0, acc); }
    part[(size_t)w * r64 + (size_t)tile * 64 + lane] = acc[0];
  } else {
    const float* xp[NG]; v4f a[NG]; mma_zero(a);
#pragma unroll
    for (int g = 0; g < NG; ++g) xp[g] = x + (size_t)min(4 * g + (lane & 3), t - 1) * d + 4 * (lane >> 2);
    for (int ku = k0; ku < k1; ku += 2) {
      const bool two = ku + 1 < k1; const int kv = two ? ku + 1 : ku;
      const UnitRaw<RF> r0 = unit_load<RF>(q, tile, ku, lane); XGrp<NG> x0, x1; unit_x_load(xp, ku, x0);
      const UnitRaw<RF> r1 = unit_load<RF>(q, tile, kv, lane); unit_x_load(xp, kv, x1);
      unit_mma<RF, NG>(q, r0, ku, x0, a);
      if (two) unit_mma<RF, NG>(q, r1, kv, x1, a);
    }
#pragma unroll
    for (int ti = 0; ti < 4 * NG; ++ti) if (ti < t) part[((size_t)w * t + ti) * r64 + (size_t)tile * 64 + lane] = a[ti >> 2][ti & 3];
  }
}

#define PYRE_MOE_GU_NZMAX 2
static bool moe_idot() { static const bool on = !(getenv("PYRE_MOE_IDOT") && atoi(getenv("PYRE_MOE_IDOT")) == 0); return on; }
bool pyre_moe_takes_digits(const MoeDev& m) { return moe_idot() && m.gate_e.fmt == FMT_IQ3_S && m.sh_gate.fmt == FMT_IQ3_S; }
int pyre_moe_router_shares_launch(pyre_ctx* ctx, const char* name, const QMatDev& router, const float* x, int t, int nw, int upw, float* part, uint32_t* dgx) {
  const int d = (int)router.cols; const dim3 grid(router.tiles * nw + (dgx ? (d / 64) * t : 0));
  ProfScope ps(ctx, name, qmat_gguf_bytes(router, router.rows) + 4.0 * t * (d + (double)nw * router.tiles * 64));
#define SHARES_GO(RF) do { if (t == 1) hipLaunchKernelGGL((k_moe_router_shares<RF, 0>), grid, dim3(64), 0, ctx->stream, router, x, t, d, nw, upw, part, dgx); \
                         else if (t <= 4) hipLaunchKernelGGL((k_moe_router_shares<RF, 1>), grid, dim3(64), 0, ctx->stream, router, x, t, d, nw, upw, part, dgx); \
                         else hipLaunchKernelGGL((k_moe_router_shares<RF, 2>), grid, dim3(64), 0, ctx->stream, router, x, t, d, nw, upw, part, dgx); } while (0)
  if (t < 1 || t > 8) return pyre_fail(ctx, PYRE_E_ARG, "moe: the router's shares are for 1..8 tokens");
  if (router.fmt == FMT_BF16) SHARES_GO(FMT_BF16);
  else if (router.fmt == FMT_F32) SHARES_GO(FMT_F32);
#undef SHARES_GO
  else return pyre_fail(ctx, PYRE_E_TYPE, "moe: the router's shares are for f32 and bf16 matrices");
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
static bool router_shares_ok(const MoeDev& m) { int nw, upw; pyre_gemv_plan(m.router, &nw, &upw); return (m.router.fmt == FMT_BF16 || m.router.fmt == FMT_F32) && nw <= 16; }
static size_t router_floats(const MoeDev& m) { int nw, upw; pyre_gemv_plan(m.router, &nw, &upw); const size_t sh = (size_t)nw * m.router.tiles * 64; return 8 * (sh > (size_t)m.n_exp ? sh : (size_t)m.n_exp); }      // logits, or the shares of them
size_t pyre_moe_work_bytes(const MoeDev& m) {
  size_t hs = (size_t)(m.ff > m.sf ? m.ff : m.sf), k1 = m.top_k + 1;
  return 256 * 11 + sizeof(float) * (router_floats(m) + 8 * (size_t)m.top_k * 2 + 8 + 8 * k1 * hs * 2 * PYRE_MOE_GU_NZMAX + 8 * k1 * (size_t)m.d + 8 * PYRE_MOE_GROUPS * (size_t)m.d + 8 * (size_t)(m.d / 64) * DGX_STRIDE + 8 * k1 * (hs / 64) * DGX_STRIDE);
}
void pyre_moe_work_carve(const MoeDev& m, void* base, MoeWork* w) {
  uint8_t* p = (uint8_t*)base; auto take = [&](size_t n) { void* r = p; p += (n + 255) & ~(size_t)255; return r; };
  size_t hs = (size_t)(m.ff > m.sf ? m.ff : m.sf), k1 = m.top_k + 1;
  w->logits = (float*)take(4 * router_floats(m)); w->sel_idx = (int32_t*)take(4 * 8 * (size_t)m.top_k); w->sel_w = (float*)take(4 * 8 * (size_t)m.top_k);
  w->sg = (float*)take(4 * 8); w->h = (float*)take(4 * 8 * k1 * hs * 2 * PYRE_MOE_GU_NZMAX); w->partial = (float*)take(4 * 8 * k1 * (size_t)m.d);
  w->parts = (float*)take(4 * 8 * PYRE_MOE_GROUPS * (size_t)m.d);
  w->dgx = (uint32_t*)take(4 * 8 * (size_t)(m.d / 64) * DGX_STRIDE);
  w->dgh = (uint32_t*)take(4 * 8 * k1 * (hs / 64) * DGX_STRIDE);
}

#define MOE_FMT_DISPATCH(fmt, CALL) \
  switch (fmt) { case FMT_F32: { constexpr int F = FMT_F32; CALL; } break; case FMT_F16: { constexpr int F = FMT_F16; CALL; } break; case FMT_BF16: { constexpr int F = FMT_BF16; CALL; } break; \
    case FMT_Q8_0: { constexpr int F = FMT_Q8_0; CALL; } break; case FMT_Q4_K: { constexpr int F = FMT_Q4_K; CALL; } break; case FMT_IQ2_XS: { constexpr int F = FMT_IQ2_XS; CALL; } break; \
    case FMT_C4: { constexpr int F = FMT_C4; CALL; } break; case FMT_C8: { constexpr int F = FMT_C8; CALL; } break; \
    default: { constexpr int F = FMT_IQ3_S; CALL; } break; }

static bool moe_idot_gu_only() { static const bool on = getenv("PYRE_MOE_IDOT") && atoi(getenv("PYRE_MOE_IDOT")) == 1; return on; }
// K parts of the gate/up dot products (a property of the matrices, so that every window length gives a token the
// same bits) and whether a window of t tokens launches one workgroup per part: only a single token does, whose
// tiles x (k+1) workgroups would leave most of the chip idle.
int pyre_moe_gu_parts(const MoeDev& m) {
  static const bool off = getenv("PYRE_MOE_GU_PARTS") && atoi(getenv("PYRE_MOE_GU_PARTS")) == 0;
  return (!off && m.gate_e.U % 32 == 0 && m.sh_gate.U == m.gate_e.U) ? 2 : 1;
}
// every count of experts a token up to PYRE_MOE_KMAX has its instance, larger ones the one with the count at run time
template <int K = PYRE_MOE_KMAX> static void moe_route_launch(int k, const MoeDev& m, dim3 grid, hipStream_t st, const float* lg, int32_t* sel_idx, float* sel_w, int nsl, int sstride, int tstride) {
  if constexpr (K > 0) { if (k != K) return moe_route_launch<K - 1>(k, m, grid, st, lg, sel_idx, sel_w, nsl, sstride, tstride); }
  if (nsl <= 16) hipLaunchKernelGGL((k_moe_route<K, 16>), grid, dim3(1024), 0, st, m, lg, sel_idx, sel_w, nsl, sstride, tstride);
  else if (nsl <= 32) hipLaunchKernelGGL((k_moe_route<K, 32>), grid, dim3(1024), 0, st, m, lg, sel_idx, sel_w, nsl, sstride, tstride);
  else hipLaunchKernelGGL((k_moe_route<K, 64>), grid, dim3(1024), 0, st, m, lg, sel_idx, sel_w, nsl, sstride, tstride);
}
int pyre_moe_launch(pyre_ctx* ctx, const MoeDev& m, const MoeWork& w, const float* x, int t, float* y, const RouteSrc* routed, bool in_groups) {
  if (in_groups && (y || t < 2 || !pyre_moe_groups_ok(m))) return pyre_fail(ctx, PYRE_E_ARG, "moe_ffn: group sums are for unreduced windows of 2..8 tokens with top_k <= %d", PYRE_MOE_KMAX);
  if (t < 1 || t > 8) return pyre_fail(ctx, PYRE_E_ARG, "moe_ffn: t = %d outside 1..8", t);
  if (!y && m.top_k > PYRE_MOE_KMAX) return pyre_fail(ctx, PYRE_E_SHAPE, "moe_ffn: an unreduced output needs top_k <= %d", PYRE_MOE_KMAX);
  if (routed && (routed->nsl < 1 || routed->nsl > 64 || routed->r64 < m.n_exp)) return pyre_fail(ctx, PYRE_E_ARG, "moe_ffn: %d router slices of %d rows", routed->nsl, routed->r64);
  auto mat_bytes = [](const QMatDev& q, double rows) { return qmat_gguf_bytes(q, rows); };
  const int hs = m.ff > m.sf ? m.ff : m.sf, entries = t * (m.top_k + 1);
  const uint2* g2 = (const uint2*)ctx->d_iq2xs;
  const int P = pyre_moe_gu_parts(m), nz = (P > 1 && t == 1) ? P : 1;
  // IQ3_S experts: gate/up in the integer form, on the digits the mix left beside the activations or on a launch of their own
  const bool idot = pyre_moe_takes_digits(m);
  const uint32_t* dgx = nullptr;
  // ... and the down products on the digits of h, which a window's gate/up launch leaves and a single token's down launch forms
  const bool idot_dn = idot && !moe_idot_gu_only() && m.down_e.fmt == FMT_IQ3_S && m.sh_down.fmt == FMT_IQ3_S;
  uint32_t* dgh = idot_dn ? w.dgh : nullptr;
  // the router's sums: given (a mix left them), or the shares of its GEMV's waves, which the selection adds in wave order -- a
  // workgroup a share and row tile instead of one a row tile (eight of them at 512 experts: 8.5 us) -- with the digits in the same launch
  const float* lg = w.logits; int nsl = 1, sstride = 0, tstride = m.n_exp;
  if (routed) { lg = routed->p; nsl = routed->nsl; sstride = t * routed->r64; tstride = routed->r64; }
  else if (router_shares_ok(m)) {
    int nw, upw; pyre_gemv_plan(m.router, &nw, &upw); nsl = nw; tstride = m.router.tiles * 64; sstride = t * tstride;
    int rc = pyre_moe_router_shares_launch(ctx, "moe_router", m.router, x, t, nw, upw, w.logits, idot ? w.dgx : nullptr); if (rc) return rc;
    dgx = idot ? w.dgx : nullptr;
  } else { int rc = pyre_gemv_launch(ctx, m.router, x, t, w.logits); if (rc) return rc; }
  if (idot && !dgx) {
    if (routed && routed->dgx) dgx = routed->dgx;
    else { ProfScope ps(ctx, "moe_digits", 4.0 * t * m.d * 2); hipLaunchKernelGGL(k_act_digits_eo, dim3(m.d / 64, t), dim3(64), 0, ctx->stream, x, m.d, w.dgx); PYRE_CHECK_LAUNCH(ctx); dgx = w.dgx; }
  }
  const bool a3b = t == 1 && m.gate_e.fmt == FMT_IQ3_S && m.down_e.fmt == FMT_IQ3_S && m.n_exp == 512 && m.top_k == 10 && m.d == 2048 && m.ff == 512 && m.sf == 512;          // the instances with these constants folded in
  { ProfScope ps(ctx, "moe_route_gate_up", t * (2.0 * m.top_k * mat_bytes(m.gate_e, m.ff) + 2.0 * mat_bytes(m.sh_gate, m.sf)) + 4.0 * t * (m.n_exp + 2.0 * m.d));
#define GU_ARGS(NZ) dim3(hs / 64, entries, NZ), dim3(16 * 64), 0, ctx->stream, m, lg, w.sel_idx, w.sel_w, w.sg, x, w.h, hs, g2, nsl, sstride, tstride, dgx, dgh, (const int32_t*)nullptr
#define GU_GO(PP, NZ, PRE) do { if (idot) hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, PP, PRE, false, true>), GU_ARGS(NZ)); else MOE_FMT_DISPATCH(m.gate_e.fmt, hipLaunchKernelGGL((k_moe_gu<F, 16, PP, PRE>), GU_ARGS(NZ))); } while (0)
  if (t == 1 && a3b && nsl == 32 && nz == 2) { if (idot) hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 1, false, true, true>), GU_ARGS(2)); else hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 1, false, true>), GU_ARGS(2)); }
  else if (t == 1) { GU_GO(1, nz, false); }          // the selection inside the launch; one workgroup per K part
  else {
    const bool a3bw = m.gate_e.fmt == FMT_IQ3_S && m.down_e.fmt == FMT_IQ3_S && m.n_exp == 512 && m.top_k == 10 && m.d == 2048 && m.ff == 512 && m.sf == 512;          // a window of the A3B configuration: constants folded in
    moe_route_launch(m.top_k <= PYRE_MOE_KMAX ? m.top_k : 0, m, dim3(t), ctx->stream, lg, w.sel_idx, w.sel_w, nsl, sstride, tstride);
    if (a3bw && P == 2) { if (idot) hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 2, true, true, true>), GU_ARGS(1)); else hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 2, true, true>), GU_ARGS(1)); }
    else if (P == 2) { GU_GO(2, 1, true); } else { GU_GO(1, 1, true); }
  } }
#undef GU_GO
#undef GU_ARGS
  PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "moe_down", t * (m.top_k * mat_bytes(m.down_e, m.d) + mat_bytes(m.sh_down, m.d)));
  if (in_groups) {
    const int gsz = (m.top_k + 4) / 4, last = m.top_k - min(m.top_k, (PYRE_MOE_GROUPS - 1) * gsz) + 1;          // entries of a full group, of the last (with the shared expert)
#define DOWN_G_GO(GE) MOE_FMT_DISPATCH(m.down_e.fmt, hipLaunchKernelGGL((k_moe_down_groups<F, 8, GE>), dim3(m.d / 64, t, PYRE_MOE_GROUPS), dim3(8 * 64), 0, ctx->stream, m, w.sel_idx, w.sel_w, w.sg, w.h, hs, w.parts, g2, dgh))
#define DOWN_G_ARGS dim3(m.d / 64, t, PYRE_MOE_GROUPS), dim3(8 * 64), 0, ctx->stream, m, w.sel_idx, w.sel_w, w.sg, w.h, hs, w.parts, g2, dgh
    if (m.gate_e.fmt == FMT_IQ3_S && m.down_e.fmt == FMT_IQ3_S && m.n_exp == 512 && m.top_k == 10 && m.d == 2048 && m.ff == 512 && m.sf == 512) {          // the A3B configuration: constants folded in
      if (idot_dn) hipLaunchKernelGGL((k_moe_down_groups<FMT_IQ3_S, 8, 3, true, true>), DOWN_G_ARGS); else hipLaunchKernelGGL((k_moe_down_groups<FMT_IQ3_S, 8, 3, true>), DOWN_G_ARGS);
    } else if (idot_dn) { if (gsz <= 3 && last <= 3) hipLaunchKernelGGL((k_moe_down_groups<FMT_IQ3_S, 8, 3, false, true>), DOWN_G_ARGS); else hipLaunchKernelGGL((k_moe_down_groups<FMT_IQ3_S, 8, PYRE_MOE_GMAX, false, true>), DOWN_G_ARGS); }
    else if (gsz <= 3 && last <= 3) { DOWN_G_GO(3); } else { DOWN_G_GO(PYRE_MOE_GMAX); }
#undef DOWN_G_ARGS
#undef DOWN_G_GO
  }
#define DOWN_ARGS dim3(m.d / 64, entries), dim3(8 * 64), 0, ctx->stream, m, w.sel_idx, w.h, hs, w.partial, g2, dgh, (const int32_t*)nullptr
  else if (a3b && nz == 2) { if (idot_dn) hipLaunchKernelGGL((k_moe_down<FMT_IQ3_S, 8, 2, true, true>), DOWN_ARGS); else hipLaunchKernelGGL((k_moe_down<FMT_IQ3_S, 8, 2, true>), DOWN_ARGS); }
  else if (idot_dn) { if (nz == 1) hipLaunchKernelGGL((k_moe_down<FMT_IQ3_S, 8, 1, false, true>), DOWN_ARGS); else hipLaunchKernelGGL((k_moe_down<FMT_IQ3_S, 8, 2, false, true>), DOWN_ARGS); }
  else if (nz == 1) { MOE_FMT_DISPATCH(m.down_e.fmt, hipLaunchKernelGGL((k_moe_down<F, 8, 1>), DOWN_ARGS)); }
  else { MOE_FMT_DISPATCH(m.down_e.fmt, hipLaunchKernelGGL((k_moe_down<F, 8, 2>), DOWN_ARGS)); } }
#undef DOWN_ARGS
  PYRE_CHECK_LAUNCH(ctx);
  if (y) {
    ProfScope ps(ctx, "moe_sum", 4.0 * t * m.d * (m.top_k + 2));
    hipLaunchKernelGGL(k_moe_sum, dim3((m.d + 255) / 256, t), dim3(256), 0, ctx->stream, w.partial, w.sel_w, w.sg, m.d, m.top_k, y);
    PYRE_CHECK_LAUNCH(ctx);
  }
  return PYRE_OK;
}

// ---- the FFN of a block of prompt windows, the tokens grouped by expert ------------------------------------------------------
// A long prompt is run layer by layer over blocks of up to 32 windows of eight tokens (model.hip); between a layer's FFN mixes
// and the next layer the FFN of all of the block's tokens runs here: an expert's weights are fetched once for all of its
// tokens (a window by itself picks eight tokens x 10 of 512 experts and shares nothing).  A token's arithmetic is that of
// the window kernels above, in the same order (k_moe_route, k_moe_gu<.., 2, true, .., ID>, k_moe_down_groups<.., ID>): its
// bits do not depend on which path ran.  IQ3_S experts in the integer form only, gate / up rows of 32 units, expert widths
// of at most 8 units.
template <bool FIX, int NSM = 64>
__global__ __launch_bounds__(1024) void k_moe_route_blk(MoeDev m, MoeBlk b, int nsl, int r64) {
  __shared__ RouteLds rl;
  const int ti = blockIdx.x, w = ti >> 3, tw = ti & 7;
  const int n_exp = FIX ? 512 : m.n_exp, top_k = FIX ? 10 : m.top_k;
  if constexpr (FIX && NSM == 64) nsl = 32;
#ifdef PYRE_PHASE_TS
  unsigned long long ts_[8];
#endif
  route_topk<1024, NSM>(b.rpart + (size_t)w * b.wr + (size_t)tw * r64, nsl, 8 * r64, n_exp, top_k, rl ROUTE_TS_ARG);
  route_weights(top_k, rl);
  if ((int)threadIdx.x < top_k) { b.sel_idx[ti * top_k + threadIdx.x] = rl.s_idx[threadIdx.x]; b.sel_w[ti * top_k + threadIdx.x] = rl.s_w[threadIdx.x]; }
}
// A block's router logits when they do not ride on the windows' FFN mixes: grid (row tiles, groups of eight tokens), 8 waves.  The riding code of
// k_hc_up_mix_m forms a sum for every 64 columns and the selection adds them in order; here the workgroup's waves form four of them each
// (unit_mma: the same bits) and add them on the spot, so that the logits leave instead of d / 64 sums a logit (134 MB at 2048 tokens of 512
// experts).  f32 products: 34 us at 126 TFLOP/s; 74 -> 53 us, and the selection, which read the sums, 19 -> 11.
template <int RF>
__global__ __launch_bounds__(512) void k_moe_router_blk(MoeDev m, MoeBlk b, int r64) {
  __shared__ float sl[32][8][64];
  const int tile = blockIdx.x, w = blockIdx.y, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, U = m.router.U;
  const float* xp[2] = {b.x + (size_t)(w * 8 + (lane & 3)) * m.d + 4 * (lane >> 2), b.x + (size_t)(w * 8 + 4 + (lane & 3)) * m.d + 4 * (lane >> 2)};
  float v = 0.0f;          // token `wave`, row `lane`
  for (int k0 = 0; k0 < U; k0 += 32) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const int s = wave * 4 + i, ka = min(k0 + s, U - 1), kb = min(k0 + s + 1, U - 1);
      const UnitRaw<RF> r0 = unit_load<RF>(m.router, tile, ka, lane); XGrp<2> x0, x1; unit_x_load(xp, ka, x0);
      const UnitRaw<RF> r1 = unit_load<RF>(m.router, tile, kb, lane); unit_x_load(xp, kb, x1);
      v4f a0[2], a1[2]; mma_zero(a0); mma_zero(a1);
      unit_mma<RF, 2>(m.router, r0, ka, x0, a0); unit_mma<RF, 2>(m.router, r1, kb, x1, a1);
#pragma unroll
      for (int t = 0; t < 8; ++t) { sl[s][t][lane] = a0[t >> 2][t & 3]; sl[s + 1][t][lane] = a1[t >> 2][t & 3]; }
    }
    lds_barrier();
    const int n = min(32, U - k0);
    if (n == 32) {
#pragma unroll
      for (int q = 0; q < 32; ++q) v = q == 0 && k0 == 0 ? sl[0][wave][lane] : v + sl[q][wave][lane];
    } else for (int q = 0; q < n; ++q) v = q == 0 && k0 == 0 ? sl[0][wave][lane] : v + sl[q][wave][lane];
    if (k0 + 32 < U) lds_barrier();
  }
  const_cast<float*>(b.rpart)[(size_t)w * b.wr + (size_t)wave * r64 + (size_t)tile * 64 + lane] = v;
}
#define MOE_PASS 8
// the (token, choice) pairs of the block by expert: eoff[e] .. eoff[e + 1] of elist hold expert e's entries token * (k + 1) + j
// (in no particular order: a token's sums do not depend on its neighbours).  One workgroup of 1024 threads.
__global__ __launch_bounds__(1024) void k_moe_lists(MoeDev m, MoeBlk b, int T) {
  __shared__ int cnt[1024], cur[1024];
  const int tid = threadIdx.x, k = m.top_k, np = T * k;
  cnt[tid] = 0;
  __syncthreads();
  for (int p = tid; p < np; p += 1024) atomicAdd(&cnt[b.sel_idx[p]], 1);
  __syncthreads();
  const int own = cnt[tid]; int v = own;
  for (int o = 1; o < 1024; o <<= 1) { cur[tid] = v; __syncthreads(); const int a = tid >= o ? cur[tid - o] : 0; __syncthreads(); v += a; }
  cur[tid] = v - own;            // exclusive prefix
  if (tid <= m.n_exp) b.eoff[tid] = tid < m.n_exp ? v - own : np;
  __syncthreads();
  if (b.plist) {                 // the experts' entries in passes of MOE_PASS: expert << 16 | pass of the expert
    const int mine = (own + MOE_PASS - 1) / MOE_PASS; int c = mine;
    for (int o = 1; o < 1024; o <<= 1) { cnt[tid] = c; __syncthreads(); const int a = tid >= o ? cnt[tid - o] : 0; __syncthreads(); c += a; }
    if (tid == 1023) b.plist[0] = c;
    for (int i = 0; i < mine; ++i) b.plist[1 + c - mine + i] = tid << 16 | i;
  }
  for (int p = tid; p < np; p += 1024) { const int pos = atomicAdd(&cur[b.sel_idx[p]], 1); b.elist[pos] = (p / k) * (k + 1) + p % k; }
}
// What a workgroup of the two kernels below works on: blockIdx.y < n_exp: the routed expert's entries; above: eight tokens'
// entries of the shared expert.
struct BlkEntries { int n; const int32_t* list; int first; int step; };
__device__ __forceinline__ BlkEntries blk_entries(const MoeDev& m, const MoeBlk& b, int T, int ye) {
  BlkEntries e;
  if (ye < m.n_exp) { const int e0 = b.eoff[ye]; e.n = b.eoff[ye + 1] - e0; e.list = b.elist + e0; e.first = 0; e.step = 0; }
  else { const int t0 = (ye - m.n_exp) * 8; e.n = min(8, T - t0); e.list = nullptr; e.first = t0 * (m.top_k + 1) + m.top_k; e.step = m.top_k + 1; }
  return e;
}
__device__ __forceinline__ int blk_entry(const BlkEntries& e, int i) { return e.list ? e.list[i] : e.first + i * e.step; }

// f32 rows -> the matrix cores' operand, a row at a time: row r of x [n][cols] as its two f16 halves xh[r][0 / 1][cols], each
// 256-column stretch on its own power of two (the arithmetic of k_act_split, gemm_m.hip), the inverse factors in
// inv[r][cols / 256].  x2 given: the row is silu(x) * x2 (an expert's h out of its gate and up products).  gate_inp given:
// sg[r] = sigmoid(gate_inp . x[r]) as well (the shared expert's gate).  grid (n), 256 threads, a stretch a round.  Row n of
// xh is kept zero by the owner: the operand rows a pass has no token for point there.
__global__ __launch_bounds__(256) void k_blk_split(const float* __restrict__ x, const float* __restrict__ x2, int cols, uint16_t* __restrict__ xh, float* __restrict__ inv, const float* __restrict__ gate_inp, float* __restrict__ sg) {
  __shared__ float mx[2][4]; __shared__ float dp[4];
  const int r = blockIdx.x, i = threadIdx.x, wave = i >> 6, lane = i & 63;
  float dot = 0.0f;
  for (int sb = 0; sb < (cols >> 8); ++sb) {
    const int k = sb * 256 + i;
    float v = x[(size_t)r * cols + k];
    if (x2) { const float sgm = 1.0f / (1.0f + expf(-v)); v = (v * sgm) * x2[(size_t)r * cols + k]; }
    if (gate_inp) dot = fmaf(gate_inp[k], v, dot);
    float a = fabsf(v); a = a == a ? a : INFINITY;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a = fmaxf(a, __shfl_xor(a, o));
    if (lane == 0) mx[sb & 1][wave] = a;
    __syncthreads();            // (the two halves of mx take turns: one barrier a round)
    const float mv = fmaxf(fmaxf(mx[sb & 1][0], mx[sb & 1][1]), fmaxf(mx[sb & 1][2], mx[sb & 1][3]));
    int e = 0;
    if (mv > 0.0f && mv < INFINITY) { e = 140 - (int)((__float_as_uint(mv) >> 23) & 0xFF); e = e > 100 ? 100 : e; }
    const float up = __uint_as_float((uint32_t)(127 + e) << 23), dn = __uint_as_float((uint32_t)(127 - e) << 23);
    const float xs = v * up;
    const _Float16 h1 = (_Float16)xs, h2 = (_Float16)((xs - (float)h1) * 2048.0f);
    xh[((size_t)r * 2) * cols + k] = __builtin_bit_cast(unsigned short, h1); xh[((size_t)r * 2 + 1) * cols + k] = __builtin_bit_cast(unsigned short, h2);
    if (i == 0) inv[(size_t)r * (cols >> 8) + sb] = dn;
  }
  if (gate_inp) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o);
    if (lane == 0) dp[wave] = dot;
    __syncthreads();
    if (i == 0) sg[r] = 1.0f / (1.0f + expf(-(((dp[0] + dp[1]) + dp[2]) + dp[3])));
  }
}
// the sixteen operand rows of a pass for chunk c: lane (kg, r) takes the eight columns 32 s + 8 kg .. of half r & 1 of the row
// its slot r >> 1 names; the scale factors of the two slots whose sums the lane holds
__device__ __forceinline__ void load_a_rows(const uint16_t* __restrict__ p, const float* __restrict__ i0, const float* __restrict__ i1, int c, ABuf& b) {
#pragma unroll
  for (int s = 0; s < 4; ++s) b.a[s] = *(const uint4*)(p + c * 128 + s * 32);
  b.ai0 = i0[c >> 1]; b.ai1 = i1[c >> 1];
}

// The expert products of a block on the matrix cores.  DOWN = false: gate and up (blockIdx.z), grid (ff / 256, n_exp +
// ceil(T / 8), 2), operand rows of x by token, out g / u [entry][ff]; DOWN = true: grid (d / 256, same, 1), operand rows of h
// by entry, out the unreduced terms partial[entry][d].  4 waves, each with 64 rows of its expert's matrix (FMT_IQ3_S_M) of
// its own: the wave walks all of the row tile's 128-column chunks with two register buffers taking turns and writes its sums
// itself -- no shared memory, no barrier.  The workgroup's entries go through in passes of eight (sixteen operand rows); a
// weight is decoded once a pass, whatever the pass holds.
template <bool DOWN>
__global__ __launch_bounds__(256, 3) void k_moe_mm_blk(MoeDev m, MoeBlk b, int T, int zrow) {            // zrow: the operand's zero row
  const int ye = blockIdx.y; const bool shared = ye >= m.n_exp;
  const BlkEntries E = blk_entries(m, b, T, ye);
  if (E.n <= 0) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, k1 = m.top_k + 1;
  const QMatDev& W = DOWN ? (shared ? m.sh_down_m : m.down_m) : (blockIdx.z ? (shared ? m.sh_up_m : m.up_m) : (shared ? m.sh_gate_m : m.gate_m));
  const int rows = DOWN ? m.d : m.ff, kc = DOWN ? m.ff : m.d;
  const int rt = blockIdx.x * 4 + wave;            // the wave's row tile inside the expert
  if (rt * 64 >= rows) return;
  const uint16_t* opnd = DOWN ? b.hh : b.xh; const float* inv = DOWN ? b.hinv : b.xinv;
  float* out = DOWN ? b.partial : (blockIdx.z ? b.u : b.g);
  const int tile = (shared ? 0 : ye * (rows >> 6)) + rt;
  const int K128 = kc >> 7, nsb = kc >> 8;
  const NibK nk = nib_consts();
  const int kg = lane >> 4, r = lane & 15, slot = r >> 1, half = r & 1, q = lane >> 4;
  for (int i0 = 0; i0 < E.n; i0 += 8) {
    const int np = min(8, E.n - i0);
    auto row_of = [&](int sl) { const int en = blk_entry(E, i0 + sl); return DOWN ? en : en / k1; };
    const size_t myrow = slot < np ? (size_t)row_of(slot) : (size_t)zrow;
    const uint16_t* ap = opnd + (myrow * 2 + half) * kc + kg * 8;
    const bool on0 = 2 * q < np, on1 = 2 * q + 1 < np;
    const float* ip0 = inv + (size_t)(on0 ? row_of(2 * q) : 0) * nsb;            // (a slot without a token reads some row's factors: its sums are never written)
    const float* ip1 = inv + (size_t)(on1 ? row_of(2 * q + 1) : 0) * nsb;
    v4f tot[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) tot[g] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    WBuf<4> w0, w1; ABuf a0, a1;
    load_a_rows(ap, ip0, ip1, 0, a0); load_w<4>(W, tile * 4, 0, lane, K128, w0);
    for (int c = 0; c < K128; c += 2) {
      if (c + 1 < K128) { load_a_rows(ap, ip0, ip1, c + 1, a1); load_w<4>(W, tile * 4, c + 1, lane, K128, w1); }
      __builtin_amdgcn_sched_barrier(0);
      chunk_mac<4>(w0, a0, c, nk, tot);
      __builtin_amdgcn_sched_barrier(0);
      if (c + 2 < K128) { load_a_rows(ap, ip0, ip1, c + 2, a0); load_w<4>(W, tile * 4, c + 2, lane, K128, w0); }
      __builtin_amdgcn_sched_barrier(0);
      if (c + 1 < K128) chunk_mac<4>(w1, a1, c + 1, nk, tot);
      __builtin_amdgcn_sched_barrier(0);
    }
    // lane (q, j) holds, for row group g, token slot 2q (halves h1, h2 * 2^11 in rows 0, 1 of its four) and slot 2q + 1
    float* o0 = on0 ? out + (size_t)blk_entry(E, i0 + 2 * q) * rows + rt * 64 + r : nullptr;
    float* o1 = on1 ? out + (size_t)blk_entry(E, i0 + 2 * q + 1) * rows + rt * 64 + r : nullptr;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (o0) o0[g * 16] = tot[g][0] + tot[g][1] * (1.0f / 2048.0f);
      if (o1) o1[g * 16] = tot[g][2] + tot[g][3] * (1.0f / 2048.0f);
    }
  }
}
// The same products where an expert has many tokens: the workgroup takes up to TG groups of eight entries through together, so
// that a weight is decoded once for all of them (k_moe_mm_blk decodes it again every eight entries: at 2048 tokens, forty
// entries an expert, 710 us a layer for gate and up).  A chunk of the groups' operand rows (16 rows x 256 bytes a group) goes
// from memory straight into shared memory once for the four waves, a row's sixteen pieces in the order piece ^ row, so that
// neither the gather (whole rows) nor the reads (sixteen rows, one piece each) meet on a bank.  Same sums in the same order.
template <bool DOWN, int TG>
__global__ __launch_bounds__(256, 2) void k_moe_mm_many(MoeDev m, MoeBlk b, int T, int zrow) {
  __shared__ __align__(16) uint4 la[2][TG][256];
  extern __shared__ __align__(16) float li[];          // [TG][super-blocks][8]
  const int ye = blockIdx.y, k1 = m.top_k + 1; const bool shared = ye >= m.n_exp;
  BlkEntries E;
  if (!shared) { const int e0 = b.eoff[ye]; E.n = b.eoff[ye + 1] - e0; E.list = b.elist + e0; E.first = 0; E.step = 0; }
  else { const int t0 = (ye - m.n_exp) * 8 * TG; E.n = min(8 * TG, T - t0); E.list = nullptr; E.first = t0 * k1 + m.top_k; E.step = k1; }
  if (E.n <= 0) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const QMatDev& W = DOWN ? (shared ? m.sh_down_m : m.down_m) : (blockIdx.z ? (shared ? m.sh_up_m : m.up_m) : (shared ? m.sh_gate_m : m.gate_m));
  const int rows = DOWN ? m.d : m.ff, kc = DOWN ? m.ff : m.d, rt = blockIdx.x * 4 + wave;          // (rows % 256 == 0: every wave has a tile)
  const uint16_t* opnd = DOWN ? b.hh : b.xh; const float* inv = DOWN ? b.hinv : b.xinv;
  float* out = DOWN ? b.partial : (blockIdx.z ? b.u : b.g);
  const int tile = (shared ? 0 : ye * (rows >> 6)) + rt, K128 = kc >> 7, nsb = kc >> 8;
  const NibK nk = nib_consts();
  const int fr = 4 * wave + (lane >> 4), fcg = (lane & 15) ^ fr;          // the operand row and piece this lane fetches
  for (int i0 = 0; i0 < E.n; i0 += 8 * TG) {
    const int np = min(8 * TG, E.n - i0), ng = (np + 7) >> 3;
    auto row_of = [&](int sl) { const int en = blk_entry(E, i0 + sl); return DOWN ? en : en / k1; };
    uint32_t so[TG];          // byte offsets (the operand stays below 4 GB: pyre_moe_block_launch)
#pragma unroll
    for (int u = 0; u < TG; ++u) { const int sl = u * 8 + (fr >> 1); so[u] = (((uint32_t)(sl < np ? row_of(sl) : zrow) * 2 + (fr & 1)) * (uint32_t)kc + fcg * 8) * 2; }
    if (i0 > 0) __syncthreads();
    for (int i = threadIdx.x; i < ng * 8 * nsb; i += 256) { const int sl = i / nsb, sb = i - sl * nsb; li[((sl >> 3) * nsb + sb) * 8 + (sl & 7)] = sl < np ? inv[(size_t)row_of(sl) * nsb + sb] : 0.0f; }
    auto fetch = [&](int c, int buf) {
#pragma unroll
      for (int u = 0; u < TG; ++u) if (u < ng) lds_fetch16((const uint8_t*)opnd + so[u] + c * 256, &la[buf][u][wave * 64]);
    };
    v4f tot[TG][4];
#pragma unroll
    for (int u = 0; u < TG; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g) tot[u][g] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    WBuf<4> wb; fetch(0, 0); load_w<4>(W, tile * 4, 0, lane, K128, wb);
    lds_fetch_barrier();
    for (int c = 0; c < K128; ++c) {
      v8h a[4];
      auto read_a = [&](int u) {
#pragma unroll
        for (int s = 0; s < 4; ++s) a[s] = __builtin_bit_cast(v8h, la[c & 1][u][r * 16 + ((s * 4 + q) ^ r)]);
      };
      read_a(0);
      WDec wd[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) decode_chunk(wb.w[g], wb.h[g], c, nk, wd[g]);
      if (c + 1 < K128) { fetch(c + 1, (c + 1) & 1); load_w<4>(W, tile * 4, c + 1, lane, K128, wb); }
#pragma unroll
      for (int u = 0; u < TG; ++u) if (u < ng) {
        v4f acc[4]; const float2 ai = *(const float2*)&li[(u * nsb + (c >> 1)) * 8 + 2 * q];
        multi_mfma<4>(wd, a, acc);
        __builtin_amdgcn_sched_barrier(0);
        if (u + 1 < TG) read_a(u + 1);          // (behind the instructions that read the registers, in flight beside the scaling)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 4; ++g) scale_add(acc[g], wd[g].d, ai.x, ai.y, tot[u][g]);
      }
      lds_fetch_barrier();
    }
#pragma unroll
    for (int u = 0; u < TG; ++u) if (u < ng) {
      const int s0 = u * 8 + 2 * q;
      float* o0 = s0 < np ? out + (size_t)blk_entry(E, i0 + s0) * rows + rt * 64 + r : nullptr;
      float* o1 = s0 + 1 < np ? out + (size_t)blk_entry(E, i0 + s0 + 1) * rows + rt * 64 + r : nullptr;
#pragma unroll
      for (int g = 0; g < 4; ++g) { if (o0) o0[g * 16] = halves0(tot[u][g]); if (o1) o1[g * 16] = halves1(tot[u][g]); }
    }
  }
}
// the four group sums of every token (moe_out_value's groups, folded as k_moe_down_groups folds them) into the token's
// window: grid (d / 256, T), thread = row
__global__ __launch_bounds__(256) void k_moe_groups_blk(MoeDev m, MoeBlk b, int T) {
  const int r = blockIdx.x * 256 + threadIdx.x, ti = blockIdx.y, k = m.top_k, d = m.d, gsz = (k + 4) / 4;
  if (r >= d) return;
  const float* pt = b.partial + (size_t)ti * (k + 1) * d + r;
  float* out = b.parts + (size_t)(ti >> 3) * PYRE_MOE_GROUPS * 8 * d + (size_t)(ti & 7) * d + r;
#pragma unroll
  for (int q = 0; q < PYRE_MOE_GROUPS; ++q) {
    const int j0 = min(k, q * gsz), nr = min(k, j0 + gsz) - j0;
    float o = 0.0f;
    for (int e = 0; e < nr; ++e) o = fmaf(b.sel_w[ti * k + j0 + e], pt[(size_t)(j0 + e) * d], o);
    if (q == PYRE_MOE_GROUPS - 1) o = fmaf(pt[(size_t)k * d], b.sg[ti], o);            // the shared expert comes last
    out[(size_t)q * 8 * d] = o;
  }
}

static bool is_m(const QMatDev& q) { return q.fmt == FMT_IQ3_S_M && q.mq && q.mh; }
bool pyre_moe_block_ok(const MoeDev& m) {
  return is_m(m.gate_m) && is_m(m.up_m) && is_m(m.down_m) && is_m(m.sh_gate_m) && is_m(m.sh_up_m) && is_m(m.sh_down_m) && m.d % 256 == 0 && m.ff % 256 == 0 && m.sf == m.ff &&
         m.n_exp <= 1023 && pyre_moe_groups_ok(m);
}
size_t pyre_moe_block_bytes(const MoeDev& m, int T) {
  const size_t hs = (size_t)m.ff, k1 = m.top_k + 1, n = (size_t)T, ne = n * k1;
  return 256 * 12 + 4 * (2 * n * m.top_k + n + 1024 + n * m.top_k + 2 * ne * hs + ne * (size_t)m.d + ne * (hs / 256) + n * (m.d / 256)) + 2 * (2 * (n + 1) * m.d + 2 * (ne + 1) * hs);
}
void pyre_moe_block_carve(const MoeDev& m, int T, void* base, MoeBlk* b) {
  uint8_t* p = (uint8_t*)base; auto take = [&](size_t n) { void* r = p; p += (n + 255) & ~(size_t)255; return r; };
  const size_t hs = (size_t)m.ff, k1 = m.top_k + 1, n = (size_t)T, ne = n * k1;
  b->sel_idx = (int32_t*)take(4 * n * m.top_k); b->sel_w = (float*)take(4 * n * m.top_k); b->sg = (float*)take(4 * n); b->eoff = (int32_t*)take(4 * 1024); b->elist = (int32_t*)take(4 * n * m.top_k);
  b->g = (float*)take(4 * ne * hs); b->u = (float*)take(4 * ne * hs); b->partial = (float*)take(4 * ne * (size_t)m.d);
  b->xh = (uint16_t*)take(2 * 2 * (n + 1) * m.d); b->xinv = (float*)take(4 * n * (m.d / 256));
  b->hh = (uint16_t*)take(2 * 2 * (ne + 1) * hs); b->hinv = (float*)take(4 * ne * (hs / 256));
}
// the rows no token owns: row T of xh, row T * (top_k + 1) of hh (once, when the block's scratch is made: for the largest T)
int pyre_moe_block_zero_rows(pyre_ctx* ctx, const MoeDev& m, const MoeBlk& b, int T) {
  const size_t hs = (size_t)m.ff, ne = (size_t)T * (m.top_k + 1);
  PYRE_HIP(ctx, hipMemsetAsync(b.xh + (size_t)2 * T * m.d, 0, 2 * 2 * (size_t)m.d, ctx->stream));
  PYRE_HIP(ctx, hipMemsetAsync(b.hh + 2 * ne * hs, 0, 2 * 2 * hs, ctx->stream));
  return PYRE_OK;
}
// The first T of T_router tokens (the router's logits are formed for all of them, r64 floats a token); T_max: the T the scratch was carved and its zero rows were set for (x readable up to the next multiple of eight rows)
int pyre_moe_block_launch(pyre_ctx* ctx, const MoeDev& m, const MoeBlk& b, int T, int T_router, int T_max, int r64) {
  if (!pyre_moe_block_ok(m) || T < 0 || T > T_router || T_router < 1 || T_router > T_max || (size_t)T_max * (m.top_k + 1) * m.ff * 4 >= (1ull << 32) || (size_t)T_max * m.d * 4 >= (1ull << 32) || m.d > 4096 || r64 < m.n_exp) return pyre_fail(ctx, PYRE_E_ARG, "moe block: unsupported shape (T = %d)", T);
  const int hs = m.ff, ny = m.n_exp + (T + 7) / 8, ne = T * (m.top_k + 1), ne_max = T_max * (m.top_k + 1);
  const bool fix = m.n_exp == 512 && m.top_k == 10;
  // Groups of eight entries that share an expert's decoding, by the mean entries an expert.  Gate / up + down, us, 512 experts top 10 of
  // width 512: 64 tokens (mean 1.2) 168 with one, 172 with two; 104 (2.0) 199, 189; 208 (4.1) 225 with two, 230 with four; 312 (6.1)
  // 262, 255; 520 (10) 320, 294; 2040 (40) 738 with four, 769 with six.  128 experts top 8: 104 (6.5) 92 with two, 101 with four; 160
  // (10) 119, 109; 1648 (103) 535 with four, 585 with six.
  const int mean = T * m.top_k / m.n_exp, tg = mean <= 1 ? 1 : (mean <= 6 ? 2 : 4);
#define MM_MANY(DN, TG, GX, GZ, ZR, KC) hipLaunchKernelGGL((k_moe_mm_many<DN, TG>), dim3(GX, m.n_exp + (T + 8 * TG - 1) / (8 * TG), GZ), dim3(256), (size_t)TG * 8 * (KC / 256) * 4, ctx->stream, m, b, T, ZR)
#define MM_GO(DN, GX, GZ, ZR, KC) do { if (tg == 1) hipLaunchKernelGGL(k_moe_mm_blk<DN>, dim3(GX, ny, GZ), dim3(256), 0, ctx->stream, m, b, T, ZR); else if (tg == 2) MM_MANY(DN, 2, GX, GZ, ZR, KC); else MM_MANY(DN, 4, GX, GZ, ZR, KC); } while (0)
  {
    if (m.router.U != m.d / 64 || m.router.tiles * 64 > r64 || (m.router.fmt != FMT_BF16 && m.router.fmt != FMT_F32)) return pyre_fail(ctx, PYRE_E_ARG, "moe block: router of %d units, format %d", m.router.U, m.router.fmt);
    ProfScope ps(ctx, "moe_block_router", qmat_gguf_bytes(m.router, m.router.rows) + 4.0 * T * (m.d + (double)r64));
    if (m.router.fmt == FMT_BF16) hipLaunchKernelGGL(k_moe_router_blk<FMT_BF16>, dim3(m.router.tiles, (T_router + 7) / 8), dim3(512), 0, ctx->stream, m, b, r64);
    else hipLaunchKernelGGL(k_moe_router_blk<FMT_F32>, dim3(m.router.tiles, (T_router + 7) / 8), dim3(512), 0, ctx->stream, m, b, r64);
    PYRE_CHECK_LAUNCH(ctx);
  }
  if (T == 0) return PYRE_OK;
  { ProfScope ps(ctx, "moe_block_route", 4.0 * T * m.n_exp);
    if (fix) hipLaunchKernelGGL((k_moe_route_blk<true, 1>), dim3(T), dim3(1024), 0, ctx->stream, m, b, 1, r64); else hipLaunchKernelGGL((k_moe_route_blk<false, 1>), dim3(T), dim3(1024), 0, ctx->stream, m, b, 1, r64);
    hipLaunchKernelGGL(k_moe_lists, dim3(1), dim3(1024), 0, ctx->stream, m, b, T);
    hipLaunchKernelGGL(k_blk_split, dim3(T), dim3(256), 0, ctx->stream, b.x, (const float*)nullptr, m.d, b.xh, b.xinv, m.sh_gate_inp, b.sg); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "moe_block_gate_up", 2.0 * m.n_exp * qmat_gguf_bytes(m.gate_e, m.ff) + 2.0 * qmat_gguf_bytes(m.sh_gate, m.sf));
    MM_GO(false, (hs + 255) / 256, 2, T_max, m.d);
    hipLaunchKernelGGL(k_blk_split, dim3(ne), dim3(256), 0, ctx->stream, (const float*)b.g, (const float*)b.u, hs, b.hh, b.hinv, (const float*)nullptr, (float*)nullptr); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "moe_block_down", (double)m.n_exp * qmat_gguf_bytes(m.down_e, m.d) + qmat_gguf_bytes(m.sh_down, m.d));
    MM_GO(true, (m.d + 255) / 256, 1, ne_max, hs);
#undef MM_GO
    hipLaunchKernelGGL(k_moe_groups_blk, dim3((m.d + 255) / 256, T), dim3(256), 0, ctx->stream, m, b, T); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}

// k_moe_gu<.., PRE> (both K parts in the workgroup) and k_moe_down with up to eight of an expert's tokens through together, four a matrix
// instruction (unit_mma): a weight is decoded once for them.  grid (row tiles, groups of eight of the shared expert's tokens + passes of
// eight of an expert's): one expert may have every token (a prompt whose tokens all take the same ten experts ran its 25 passes one
// behind the other on eleven workgroups a row tile: 423 us), so the passes are workgroups, not a loop.
// A K range is cut into the shares k_moe_gu / k_moe_down give their waves; here a wave walks SW of them, a unit of weights and
// activations fetched while the one before it is consumed (straight on into the next row tile or matrix), and the shares meet in
// k_moe_gu's order, so a token's bits are a window's.  What bounds it is the issue of decoding and f32 products: 200 tokens of A3B in Q4_K, ten
// experts with every token, gate / up and down 423 + 195 us -> 121 + 61 (18 GFLOP at 126 TFLOP/s: 110).
// The rows xp points at times nj row tiles: tile(j, Q) names job j's matrix and tile; the shares' sums -> red [share][4 NG][64], then done(j).
template <int FMT, int NG, int SW, class TF, class DF>
__device__ __forceinline__ void rows_jobs(int nj, TF tile, const float* const (&xp)[NG], int s0, int upw, int U, int lane, float* red, DF done) {
  const int k0 = min(U, s0 * upw), k1 = min(U, (s0 + SW) * upw);
  UnitRaw<FMT> r0, r1; XGrp<NG> x0, x1; v4f a[NG]; mma_zero(a);
  auto store = [&](int sh) {
#pragma unroll
    for (int t = 0; t < 4 * NG; ++t) red[(sh * 4 * NG + t) * 64 + lane] = a[t >> 2][t & 3];
    mma_zero(a); };
  auto fetch = [&](int j, int k, UnitRaw<FMT>& r, XGrp<NG>& x) { QMatDev Q; const int t = tile(min(j, nj - 1), Q); r = unit_load<FMT>(Q, t, k, lane); unit_x_load(xp, k, x); };
  auto finish = [&](int j) {
    for (int sh = s0; sh < s0 + SW; ++sh) if (sh * upw >= U) store(sh);          // (shares past the end: zero)
    lds_barrier(); done(j); lds_barrier(); };
  int sh = s0, left = upw;
  auto step = [&](int j, int k, const UnitRaw<FMT>& r, const XGrp<NG>& x) {
    QMatDev Q; tile(j, Q);
    unit_mma<FMT, NG>(Q, r, k, x, a);
    if (--left == 0 || k + 1 == U) { store(sh); ++sh; left = upw; }
    if (k + 1 == k1) { finish(j); sh = s0; left = upw; } };
  if (k0 >= k1) { for (int j = 0; j < nj; ++j) finish(j); return; }
  auto next = [&](int& j, int& k) { if (++k == k1) { k = k0; ++j; } };
  int j = 0, k = k0; fetch(0, k0, r0, x0);
  while (j < nj) {
    int j2 = j, k2 = k; next(j2, k2);
    fetch(j2, k2, r1, x1);
    step(j, k, r0, x0);
    if (j2 >= nj) break;
    j = j2; k = k2; next(j, k);
    fetch(j, k, r0, x0);
    step(j2, k2, r1, x1);
  }
}
// what a workgroup multiplies: n entries of `expert` (list), or those of n tokens from t0 of the shared expert (-1)
struct RowsPass { int expert, n, t0; const int32_t* list; };
__device__ __forceinline__ RowsPass rows_pass_of(const MoeDev& m, const MoeRows& w, int T) {
  const int ns = (T + MOE_PASS - 1) / MOE_PASS, p = (int)blockIdx.y - ns; RowsPass r;
  if (p < 0) { r.expert = -1; r.t0 = blockIdx.y * MOE_PASS; r.n = min(MOE_PASS, T - r.t0); r.list = nullptr; return r; }
  if (p >= w.plist[0]) { r.expert = 0; r.t0 = 0; r.n = 0; r.list = nullptr; return r; }
  const int e = w.plist[1 + p], i0 = (e & 0xFFFF) * MOE_PASS; r.expert = e >> 16; r.t0 = 0;
  const int e0 = w.eoff[r.expert]; r.n = min(MOE_PASS, w.eoff[r.expert + 1] - e0 - i0); r.list = w.elist + e0 + i0; return r;
}
// passes of T tokens' routed entries at most
static int moe_passes(const MoeDev& m, int T) { const int ne = T * m.top_k; return std::min(ne, m.n_exp + ne / MOE_PASS); }
template <int FMT, int NP, int NG>
__device__ __forceinline__ void gu_pass(const QMatDev& Qg, const QMatDev& Qu, int tile, const float* __restrict__ x, int d, const int32_t* __restrict__ list, int first, int k1, int n, float* __restrict__ h, int hstride, float* red) {
  const int tid = threadIdx.x, t = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, upw = (Qg.U + 16 * NP - 1) / (16 * NP);
  const float* xp[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) { const int i = min(4 * g + (lane & 3), n - 1), e = list ? list[i] : first + i * k1; xp[g] = x + (size_t)(e / k1) * d + 4 * (lane >> 2); }
  float gate = 0.0f;          // the thread's row of entry t
  rows_jobs<FMT, NG, 2 * NP>(2, [&](int j, QMatDev& Q) { Q = pick_mat(j == 0, Qg, Qu); return tile; }, xp, t * 2 * NP, upw, Qg.U, lane, red, [&](int j) {
    if (t >= n) return;
    float v = 0.0f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {          // share q of part p is q * NP + p
      float part = red[(p * 4 * NG + t) * 64 + lane];
#pragma unroll
      for (int q = 1; q < 16; ++q) part += red[((q * NP + p) * 4 * NG + t) * 64 + lane];
      v = p == 0 ? part : v + part;
    }
    if (j == 0) { gate = v; return; }
    const float s = 1.0f / (1.0f + expf(-gate)); const int e = list ? list[t] : first + t * k1;
    h[(size_t)e * hstride + blockIdx.x * 64 + lane] = (gate * s) * v; });
}
template <int FMT, int NP>
__global__ __launch_bounds__(512, 4) void k_moe_gu_rows(MoeDev m, MoeRows w, const float* __restrict__ x, int hstride, int T) {
  __shared__ float red[16 * NP * 8 * 64];
  const RowsPass P = rows_pass_of(m, w, T); const int n = P.n, t0 = P.t0, k1 = m.top_k + 1; const bool shared = P.expert < 0;
  if (n <= 0 || (int)blockIdx.x * 64 >= (shared ? m.sf : m.ff)) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const QMatDev Qg = pick_mat(shared, m.sh_gate, m.gate_e), Qu = pick_mat(shared, m.sh_up, m.up_e);
  const int tile = (shared ? 0 : P.expert * (m.ff >> 6)) + blockIdx.x, first = t0 * k1 + m.top_k;
  if (n > 4) gu_pass<FMT, NP, 2>(Qg, Qu, tile, x, m.d, P.list, first, k1, n, w.h, hstride, red); else gu_pass<FMT, NP, 1>(Qg, Qu, tile, x, m.d, P.list, first, k1, n, w.h, hstride, red);
  if (!shared || blockIdx.x) return;
  for (int t = 0; t < n; ++t) {          // the shared expert's gate of the group's tokens: the sums of k_moe_gu's sixteen waves
    const float* xt = x + (size_t)(t0 + t) * m.d; float p[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      for (int ib = tid + 512 * i; ib < m.d; ib += 1024) p[i] = fmaf(m.sh_gate_inp[ib], xt[ib], p[i]);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) p[i] += __shfl_xor(p[i], o);
      if (lane == 0) red[wave + 8 * i] = p[i];
    }
    __syncthreads();
    if (tid == 0) { float tot = 0.0f; for (int q = 0; q < 16; ++q) tot += red[q]; w.sg[t0 + t] = 1.0f / (1.0f + expf(-tot)); }
    __syncthreads();
  }
}
// grid (row tiles / MOE_DOWN_TILES, ..): four row tiles a workgroup
#define MOE_DOWN_TILES 4
template <int FMT, int NG>
__device__ __forceinline__ void down_pass(const QMatDev& D, int tile0, int row0, int nj, const float* __restrict__ h, float* __restrict__ partial, int d, const int32_t* __restrict__ list, int first, int k1, int n, int hstride, float* red) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, upw = (D.U + 7) / 8;
  const float* xp[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) { const int i = min(4 * g + (lane & 3), n - 1), e = list ? list[i] : first + i * k1; xp[g] = h + (size_t)e * hstride + 4 * (lane >> 2); }
  rows_jobs<FMT, NG, 2>(nj, [&](int j, QMatDev& Q) { Q = D; return tile0 + j; }, xp, wave * 2, upw, D.U, lane, red, [&](int j) {
    for (int t = wave; t < n; t += 4) {
      float sum = red[t * 64 + lane];
#pragma unroll
      for (int q = 1; q < 8; ++q) sum += red[(q * 4 * NG + t) * 64 + lane];
      const int e = list ? list[t] : first + t * k1;
      partial[(size_t)e * d + row0 + j * 64 + lane] = sum;
    } });
}
template <int FMT>
__global__ __launch_bounds__(256, 4) void k_moe_down_rows(MoeDev m, MoeRows w, int hstride, int T) {
  __shared__ float red[8 * 8 * 64];
  const RowsPass P = rows_pass_of(m, w, T); const int n = P.n, k1 = m.top_k + 1; const bool shared = P.expert < 0;
  if (n <= 0) return;
  const QMatDev D = pick_mat(shared, m.sh_down, m.down_e);
  const int r0 = blockIdx.x * MOE_DOWN_TILES, nj = min(MOE_DOWN_TILES, (m.d >> 6) - r0), tile = (shared ? 0 : P.expert * (m.d >> 6)) + r0, first = P.t0 * k1 + m.top_k;
  if (n > 4) down_pass<FMT, 2>(D, tile, r0 * 64, nj, w.h, w.partial, m.d, P.list, first, k1, n, hstride, red); else down_pass<FMT, 1>(D, tile, r0 * 64, nj, w.h, w.partial, m.d, P.list, first, k1, n, hstride, red);
}

// The windows' arithmetic (k_moe_gu / k_moe_down, the digits form for IQ3_S experts) for any number of tokens in one set of launches,
// entry by entry in the order of the experts: a prompt of a model whose experts have no matrix-core layout, and the last tokens of
// one whose experts have.  Router sums as in MoeBlk (rpart + group * wr).  parts: the group sums [group][PYRE_MOE_GROUPS][8][d], or
// null; y: their sum [token][d], or null; the unreduced terms stay in w (pyre_moe_rows_out).
size_t pyre_moe_rows_bytes(const MoeDev& m, int T) {
  const size_t hs = (size_t)(m.ff > m.sf ? m.ff : m.sf), k1 = m.top_k + 1, n = T;
  return 256 * 13 + 4 * (4 * n * m.top_k + 1 + n + 1024 + n * k1 * (hs + m.d) + n * (m.d / 64) * DGX_STRIDE + n * k1 * (hs / 64) * DGX_STRIDE);
}
void pyre_moe_rows_carve(const MoeDev& m, int T, void* base, MoeRows* w) {
  uint8_t* p = (uint8_t*)base; auto take = [&](size_t n) { void* r = p; p += (4 * n + 255) & ~(size_t)255; return r; };
  const size_t hs = (size_t)(m.ff > m.sf ? m.ff : m.sf), k1 = m.top_k + 1, n = T;
  w->sel_idx = (int32_t*)take(n * m.top_k); w->sel_w = (float*)take(n * m.top_k); w->elist = (int32_t*)take(n * m.top_k); w->sg = (float*)take(n); w->eoff = (int32_t*)take(1024); w->plist = (int32_t*)take(1 + n * m.top_k);
  w->h = (float*)take(n * k1 * hs); w->partial = (float*)take(n * k1 * m.d); w->dgx = (uint32_t*)take(n * (m.d / 64) * DGX_STRIDE); w->dgh = (uint32_t*)take(n * k1 * (hs / 64) * DGX_STRIDE);
}
bool pyre_moe_rows_ok(const MoeDev& m) { return m.top_k <= PYRE_MOE_KMAX && m.n_exp <= 1023 && m.d % 64 == 0; }
int pyre_moe_rows_launch(pyre_ctx* ctx, const MoeDev& m, const MoeRows& w, const float* x, int T, const float* rpart, size_t wr, int nsl, int r64, float* parts, float* y) {
  if (!pyre_moe_rows_ok(m) || T < 1 || T * (m.top_k + 1) > 65535 || nsl < 1 || nsl > 64 || r64 < m.n_exp) return pyre_fail(ctx, PYRE_E_ARG, "moe rows: unsupported shape (T = %d, %d router slices)", T, nsl);
  MoeBlk b{}; b.rpart = rpart; b.wr = wr; b.parts = parts; b.sel_idx = w.sel_idx; b.sel_w = w.sel_w; b.eoff = w.eoff; b.elist = w.elist; b.partial = w.partial; b.sg = w.sg; b.plist = w.plist;
  const int hs = m.ff > m.sf ? m.ff : m.sf, entries = T * (m.top_k + 1), P = pyre_moe_gu_parts(m), ns = (T + MOE_PASS - 1) / MOE_PASS;
  const uint2* g2 = (const uint2*)ctx->d_iq2xs;
  const bool idot = pyre_moe_takes_digits(m), idot_dn = idot && !moe_idot_gu_only() && m.down_e.fmt == FMT_IQ3_S && m.sh_down.fmt == FMT_IQ3_S;
  uint32_t* dgh = idot_dn ? w.dgh : nullptr;
  { ProfScope ps(ctx, "moe_rows_route", 4.0 * T * nsl * m.n_exp);
    if (nsl == 1 && m.n_exp == 512 && m.top_k == 10) hipLaunchKernelGGL((k_moe_route_blk<true, 1>), dim3(T), dim3(1024), 0, ctx->stream, m, b, nsl, r64);
    else if (nsl == 1) hipLaunchKernelGGL((k_moe_route_blk<false, 1>), dim3(T), dim3(1024), 0, ctx->stream, m, b, nsl, r64);
    else if (m.n_exp == 512 && m.top_k == 10 && nsl == 32) hipLaunchKernelGGL(k_moe_route_blk<true>, dim3(T), dim3(1024), 0, ctx->stream, m, b, nsl, r64); else hipLaunchKernelGGL(k_moe_route_blk<false>, dim3(T), dim3(1024), 0, ctx->stream, m, b, nsl, r64);
    hipLaunchKernelGGL(k_moe_lists, dim3(1), dim3(1024), 0, ctx->stream, m, b, T);
    if (idot) hipLaunchKernelGGL(k_act_digits_eo, dim3(m.d / 64, T), dim3(64), 0, ctx->stream, x, m.d, w.dgx); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "moe_rows_gate_up", T * (2.0 * m.top_k * qmat_gguf_bytes(m.gate_e, m.ff) + 2.0 * qmat_gguf_bytes(m.sh_gate, m.sf)));
#define ROWS_GU dim3(hs / 64, entries, 1), dim3(16 * 64), 0, ctx->stream, m, (const float*)nullptr, w.sel_idx, w.sel_w, w.sg, x, w.h, hs, g2, nsl, 0, 0, w.dgx, dgh, w.elist
    const bool fix = m.gate_e.fmt == FMT_IQ3_S && m.down_e.fmt == FMT_IQ3_S && m.n_exp == 512 && m.top_k == 10 && m.d == 2048 && m.ff == 512 && m.sf == 512;
    if (idot && fix && P == 2) hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 2, true, true, true>), ROWS_GU);
    else if (idot) { if (P == 2) hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 2, true, false, true>), ROWS_GU); else hipLaunchKernelGGL((k_moe_gu<FMT_IQ3_S, 16, 1, true, false, true>), ROWS_GU); }
    else if (P == 2) { MOE_FMT_DISPATCH(m.gate_e.fmt, hipLaunchKernelGGL((k_moe_gu_rows<F, 2>), dim3(hs / 64, ns + moe_passes(m, T)), dim3(512), 0, ctx->stream, m, w, x, hs, T)); }
    else { MOE_FMT_DISPATCH(m.gate_e.fmt, hipLaunchKernelGGL((k_moe_gu_rows<F, 1>), dim3(hs / 64, ns + moe_passes(m, T)), dim3(512), 0, ctx->stream, m, w, x, hs, T)); }
#undef ROWS_GU
  } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "moe_rows_down", T * (m.top_k * qmat_gguf_bytes(m.down_e, m.d) + qmat_gguf_bytes(m.sh_down, m.d)));
#define ROWS_DN dim3(m.d / 64, entries), dim3(8 * 64), 0, ctx->stream, m, w.sel_idx, w.h, hs, w.partial, g2, dgh, w.elist
    if (idot_dn) hipLaunchKernelGGL((k_moe_down<FMT_IQ3_S, 8, 1, false, true>), ROWS_DN);
    else if (idot) { MOE_FMT_DISPATCH(m.down_e.fmt, hipLaunchKernelGGL((k_moe_down<F, 8, 1>), ROWS_DN)); }          // (behind the digits form h is finished)
    else { MOE_FMT_DISPATCH(m.down_e.fmt, hipLaunchKernelGGL((k_moe_down_rows<F>), dim3((m.d / 64 + MOE_DOWN_TILES - 1) / MOE_DOWN_TILES, ns + moe_passes(m, T)), dim3(256), 0, ctx->stream, m, w, hs, T)); }
#undef ROWS_DN
    if (parts) hipLaunchKernelGGL(k_moe_groups_blk, dim3((m.d + 255) / 256, T), dim3(256), 0, ctx->stream, m, b, T);
    if (y) hipLaunchKernelGGL(k_moe_sum, dim3((m.d + 255) / 256, T), dim3(256), 0, ctx->stream, w.partial, w.sel_w, w.sg, m.d, m.top_k, y); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}

// ---- C ABI -------------------------------------------------------------------------------------------------------------
struct pyre_moe { pyre_ctx* ctx; MoeDev dv; MoeWork w; void* work; float* gate_inp; float* xy; };

extern "C" {

int pyre_moe_create(pyre_ctx* ctx, int top_k, const pyre_qmat* router, const pyre_qmat* gate_e, const pyre_qmat* up_e, const pyre_qmat* down_e,
                    const float* sh_gate_inp_host, const pyre_qmat* sh_gate, const pyre_qmat* sh_up, const pyre_qmat* sh_down, pyre_moe** out) {
  if (!ctx || !out || !router || !gate_e || !up_e || !down_e || !sh_gate_inp_host || !sh_gate || !sh_up || !sh_down) return pyre_fail(ctx, PYRE_E_ARG, "pyre_moe_create: null argument");
  *out = nullptr;
  size_t d = router->cols, E = router->rows; if (E == 0 || gate_e->rows % E) return pyre_fail(ctx, PYRE_E_SHAPE, "pyre_moe_create: gate_exps rows %zu not a multiple of %zu experts", gate_e->rows, E);
  size_t ff = gate_e->rows / E, sf = sh_gate->rows;
  if (gate_e->cols != d || up_e->cols != d || up_e->rows != E * ff || down_e->rows != E * d || down_e->cols != ff || sh_gate->cols != d || sh_up->cols != d || sh_up->rows != sf ||
      sh_down->rows != d || sh_down->cols != sf) return pyre_fail(ctx, PYRE_E_SHAPE, "pyre_moe_create: inconsistent expert tensor shapes");
  if (ff % 64 || sf % 64 || d % 64) return pyre_fail(ctx, PYRE_E_SHAPE, "pyre_moe_create: d, expert and shared widths must be multiples of 64");
  if (top_k < 1 || top_k > 32 || (size_t)top_k > E || E > 1024) return pyre_fail(ctx, PYRE_E_ARG, "pyre_moe_create: top_k %d / experts %zu unsupported", top_k, E);
  if (gate_e->dv.fmt != up_e->dv.fmt || sh_gate->dv.fmt != gate_e->dv.fmt || sh_up->dv.fmt != gate_e->dv.fmt || sh_down->dv.fmt != down_e->dv.fmt)
    return pyre_fail(ctx, PYRE_E_TYPE, "pyre_moe_create: gate/up (and shared gate/up) must share one type, down and shared down another");
  pyre_moe* m = new pyre_moe(); m->ctx = ctx;
  m->dv = MoeDev{router->dv, gate_e->dv, up_e->dv, down_e->dv, sh_gate->dv, sh_up->dv, sh_down->dv, nullptr, (int)d, (int)E, top_k, (int)ff, (int)sf};
  hipError_t e = hipMalloc((void**)&m->gate_inp, d * 4);
  if (e == hipSuccess) e = hipMemcpy(m->gate_inp, sh_gate_inp_host, d * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMalloc(&m->work, pyre_moe_work_bytes(m->dv));
  if (e == hipSuccess) e = hipMalloc((void**)&m->xy, 2 * 8 * d * 4);
  if (e != hipSuccess) { int rc = pyre_fail(ctx, PYRE_E_HIP, "pyre_moe_create: %s", hipGetErrorString(e)); delete m; return rc; }
  m->dv.sh_gate_inp = m->gate_inp; pyre_moe_work_carve(m->dv, m->work, &m->w);
  *out = m; return PYRE_OK;
}
void pyre_moe_destroy(pyre_moe* m) { if (!m) return; (void)hipStreamSynchronize(m->ctx->stream); (void)hipFree(m->gate_inp); (void)hipFree(m->work); (void)hipFree(m->xy); delete m; }

int pyre_moe_ffn_dev(pyre_ctx* ctx, pyre_moe* m, const float* x_dev, int t, float* y_dev) {
  if (!ctx || !m || !x_dev || !y_dev) return pyre_fail(ctx, PYRE_E_ARG, "pyre_moe_ffn: null argument");
  return pyre_moe_launch(ctx, m->dv, m->w, x_dev, t, y_dev);
}
int pyre_moe_ffn(pyre_ctx* ctx, pyre_moe* m, const float* x_host, int t, float* y_host, int32_t* sel_idx_host, float* sel_w_host) {
  if (!ctx || !m || !x_host || !y_host) return pyre_fail(ctx, PYRE_E_ARG, "pyre_moe_ffn: null argument");
  if (t < 1 || t > 8) return pyre_fail(ctx, PYRE_E_ARG, "pyre_moe_ffn: t = %d outside 1..8", t);
  size_t n = (size_t)t * m->dv.d * 4; float* xd = m->xy; float* yd = m->xy + 8 * (size_t)m->dv.d;
  PYRE_HIP(ctx, hipMemcpyAsync(xd, x_host, n, hipMemcpyHostToDevice, ctx->stream));
  int rc = pyre_moe_launch(ctx, m->dv, m->w, xd, t, yd); if (rc) return rc;
  PYRE_HIP(ctx, hipMemcpyAsync(y_host, yd, n, hipMemcpyDeviceToHost, ctx->stream));
  if (sel_idx_host) PYRE_HIP(ctx, hipMemcpyAsync(sel_idx_host, m->w.sel_idx, (size_t)t * m->dv.top_k * 4, hipMemcpyDeviceToHost, ctx->stream));
  if (sel_w_host) PYRE_HIP(ctx, hipMemcpyAsync(sel_w_host, m->w.sel_w, (size_t)t * m->dv.top_k * 4, hipMemcpyDeviceToHost, ctx->stream));
  PYRE_HIP(ctx, hipStreamSynchronize(ctx->stream)); return PYRE_OK;
}

}  // extern "C"
