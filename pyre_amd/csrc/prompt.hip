// The dense matrices of a prompt taken layer by layer: the hyper-connection mixes and the projections for hundreds of tokens in
// one launch each (model.hip's run_block), IQ3_S matrices in the matrix-core layout.
//
// Tokens come in groups of eight: a group is the sixteen operand rows (two f16 halves a token) of one
// v_mfma_f32_16x16x32_f16, as in gemm_m.h.  What a launch a window of eight tokens cannot do is share a decoded weight:
// decoding 128 columns of 16 rows is some sixty vector instructions, the product with one group four matrix
// instructions.  Here a wave decodes a chunk once and meets several groups with it, so the matrix cores, not the decoding,
// set the pace.  A token's sums are formed in one order whatever the groups beside it, so the cutting of a prompt into
// launches never shows in a token's bits.
#include "gemm_m.h"
#include <stdlib.h>
#include <algorithm>

namespace {

__device__ __forceinline__ float b_sigm(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ void b_scale_of(float m, float* up, float* dn) {      // m * 2^e in [2^13, 2^14); zero and non-finite maxima leave e = 0
  int e = 0;
  if (m > 0.0f && m < INFINITY) { e = 140 - (int)((__float_as_uint(m) >> 23) & 0xFF); e = e > 100 ? 100 : e; }
  *up = __uint_as_float((uint32_t)(127 + e) << 23); *dn = __uint_as_float((uint32_t)(127 - e) << 23);
}
__device__ __forceinline__ float b_nan_abs(float v) { const float a = fabsf(v); return a == a ? a : INFINITY; }
__device__ __forceinline__ void b_split(float xs, uint16_t* h1, uint16_t* h2) {
  const _Float16 a = (_Float16)xs, b = (_Float16)((xs - (float)a) * 2048.0f);
  *h1 = __builtin_bit_cast(unsigned short, a); *h2 = __builtin_bit_cast(unsigned short, b);
}
// ---- the product with a matrix of row tiles of 64 ------------------------------------------------------------------------------
// grid (row tiles / 4, groups / TG, K slices), 4 waves: wave w owns row tile 4 x + w and TG groups of eight tokens.  The groups' operand
// rows of a chunk (4 KB a group) go through shared memory once for the four waves, straight from memory, the next chunk's
// while this one's products run; a wave's codes and headers are in registers one chunk ahead.
// op: group g's operand at op + g * op_gs uint4 ([column / 8][16 rows] x 16 B); inv: eight factors a super-block (ish = 1) or a
// chunk (ish = 0) at inv + g * inv_gs.  One slice: y[token * ys + row]; several: slice z of group g's token t in
// y + ((g * slices + z) * 8 + t) * ys, for a mix that adds them in order.
// A window's launch (k_gemm_m) gives cw chunks of a slice to each of its waves and adds the waves' sums in order; the sums
// here fall in the same order, cw chunks at a time, so a token's bits are a window's.  CW1: cw = 1 (no running sum to keep).
// UNI: a token's factor is one power of two for all its columns (the mixes' operands) and meets the finished sum.
template <int TG, bool CW1, bool UNI>
__global__ __launch_bounds__(256, 2) void k_blk_gemm(QMatDev m, const uint4* __restrict__ op, size_t op_gs, const float* __restrict__ inv, int inv_gs, int ish, int cw, float* __restrict__ y, int ys, int T) {
  __shared__ __align__(16) uint4 la[2][TG][256];
  extern __shared__ __align__(16) float li[];            // [TG][the slice's super-blocks or chunks][8]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q = lane >> 4;
  const int K128 = m.cols >> 7, G = (T + 7) >> 3, g0 = blockIdx.y * TG, nz = gridDim.z, per = (K128 + nz - 1) / nz, c0 = blockIdx.z * per, c1 = min(K128, c0 + per);
  const int f0 = c0 >> ish, nf = ((c1 - 1) >> ish) - f0 + 1;
  const int tile = min((int)blockIdx.x * 4 + wave, m.tiles - 1);
  auto fetch = [&](int c, int buf) {
#pragma unroll
    for (int u = 0; u < TG; ++u) {          // 4 TG KB: a wave one KB of every group
      const uint4* src = op + (size_t)min(g0 + u, G - 1) * op_gs + (size_t)c * 256 + wave * 64 + lane;
      lds_fetch16(src, &la[buf][u][wave * 64]);
    }
  };
  for (int i = threadIdx.x; i < TG * nf * 8; i += 256) { const int u = i / (nf * 8), r = i - u * nf * 8; li[i] = inv[(size_t)min(g0 + u, G - 1) * inv_gs + f0 * 8 + r]; }
  float s0[TG][4], s1[TG][4]; v4f tot[CW1 ? 1 : TG][4];
#pragma unroll
  for (int u = 0; u < TG; ++u)
#pragma unroll
    for (int g = 0; g < 4; ++g) { s0[u][g] = 0.0f; s1[u][g] = 0.0f; if constexpr (!CW1) tot[u][g] = v4f{0.0f, 0.0f, 0.0f, 0.0f}; }
  const NibK nk = nib_consts();
  WBuf<4> wb; fetch(c0, 0); load_w<4>(m, tile * 4, c0, lane, K128, wb);
  lds_fetch_barrier();
  int left = cw;          // chunks until the running sums join
  for (int c = c0; c < c1; ++c) {
    const int buf = (c - c0) & 1;
    v8h a[4];
    auto read_a = [&](int u) {
#pragma unroll
      for (int s = 0; s < 4; ++s) a[s] = __builtin_bit_cast(v8h, la[buf][u][(s * 4 + q) * 16 + (lane & 15)]);
    };
    read_a(0);
    WDec wd[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) decode_chunk(wb.w[g], wb.h[g], c, nk, wd[g]);
    if (c + 1 < c1) { fetch(c + 1, buf ^ 1); load_w<4>(m, tile * 4, c + 1, lane, K128, wb); }
#pragma unroll
    for (int u = 0; u < TG; ++u) {
      v4f acc[4]; float2 ai = make_float2(1.0f, 1.0f); if constexpr (!UNI) ai = *(const float2*)&li[((size_t)u * nf + (c >> ish) - f0) * 8 + 2 * q];
      multi_mfma<4>(wd, a, acc);
      __builtin_amdgcn_sched_barrier(0);
      if (u + 1 < TG) read_a(u + 1);          // (behind the instructions that read the registers, in flight beside the scaling)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if constexpr (CW1) { const float d0 = UNI ? wd[g].d : wd[g].d * ai.x, d1 = UNI ? wd[g].d : wd[g].d * ai.y; s0[u][g] += fmaf(acc[g][1] * d0, 1.0f / 2048.0f, acc[g][0] * d0); s1[u][g] += fmaf(acc[g][3] * d1, 1.0f / 2048.0f, acc[g][2] * d1); }
        else scale_add(acc[g], wd[g].d, ai.x, ai.y, tot[u][g]);
      }
    }
    if constexpr (!CW1) if (--left == 0 || c + 1 == c1) {
      left = cw;
#pragma unroll
      for (int u = 0; u < TG; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) { s0[u][g] += halves0(tot[u][g]); s1[u][g] += halves1(tot[u][g]); tot[u][g] = v4f{0.0f, 0.0f, 0.0f, 0.0f}; }
    }
    lds_fetch_barrier();
  }
  if ((int)blockIdx.x * 4 + wave >= m.tiles) return;
#pragma unroll
  for (int u = 0; u < TG; ++u) {
    const int t0 = (g0 + u) * 8 + 2 * q; if (g0 + u >= G) break;
    float2 fu = make_float2(1.0f, 1.0f); if constexpr (UNI) fu = *(const float2*)&li[(size_t)u * nf * 8 + 2 * q];
    float* y0 = nz > 1 ? y + (((size_t)(g0 + u) * nz + blockIdx.z) * 8 + 2 * q) * ys : y + (size_t)t0 * ys;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = tile * 64 + g * 16 + (lane & 15);
      if (row < m.rows) { if (t0 < T) y0[row] = UNI ? s0[u][g] * fu.x : s0[u][g]; if (t0 + 1 < T) y0[ys + row] = UNI ? s1[u][g] * fu.y : s1[u][g]; }
    }
  }
}

// ---- f32 rows as operand rows: grid (columns / 256, groups), 256 threads, thread = column -----------------------------------------
// (the arithmetic of k_act_split: a 256-column stretch of a token on its own power of two)
__global__ __launch_bounds__(256) void k_blk_op_split(const float* __restrict__ x, int cols, int T, uint4* __restrict__ op, size_t op_gs, float* __restrict__ inv, int inv_gs) {
  __shared__ float mx[4][8]; __shared__ __align__(16) uint16_t st[32 * 16 * 8];
  const int sb = blockIdx.x, grp = blockIdx.y, i = threadIdx.x, k = sb * 256 + i, wave = i >> 6, lane = i & 63;
  float v[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = grp * 8 + t < T ? x[(size_t)(grp * 8 + t) * cols + k] : 0.0f;
#pragma unroll
  for (int t = 0; t < 8; ++t) { const float a = wave_max(b_nan_abs(v[t])); if (lane == 0) mx[wave][t] = a; }
  lds_barrier();
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    float up, dn; b_scale_of(fmaxf(fmaxf(mx[0][t], mx[1][t]), fmaxf(mx[2][t], mx[3][t])), &up, &dn);
    uint16_t* o = st + ((i >> 3) * 16 + 2 * t) * 8 + (i & 7); b_split(v[t] * up, o, o + 8);
    if (i == 0) inv[(size_t)grp * inv_gs + sb * 8 + t] = dn;
  }
  lds_barrier();
  uint4* dst = op + (size_t)grp * op_gs + (size_t)sb * 512;
  dst[i] = ((const uint4*)st)[i]; dst[256 + i] = ((const uint4*)st)[256 + i];
}

// ---- hyper-connection mix, first part: the pending update, sums of squares, [down ; inject] ---------------------------------------
// grid (slices of 256 CS columns, groups), 4 CS waves, a thread prepares one column of the slice for the group's tokens once
// and the waves walk every row tile with it (the launch for a window repeats the gather in each of its row tiles: at 43
// windows 72 us, here the streams are read once).  A workgroup is a chain of latencies, so its loads are all issued before the first
// barrier, and its sums leave through shared memory (adding the second pair's to what the first had stored waited for the stores):
// 301 tokens 34 -> 25 us, 2000 tokens 161 -> 112 us.  x is updated in place: an element has one reader.  Outputs per group: ssq, smx [slice][8], part [slice][8][tiles * 64].
// NP: vectors the pending update comes in -- 0 none, 1 = comb[token][d], 4 = comb[group][4][8][d], added in order.
template <int NP, int CS>
__global__ __launch_bounds__(256 * CS) void k_blk_mix_down(QMatDev m, const float* __restrict__ x_in, int in_ss, int in_ts, float* __restrict__ x_out, const float* __restrict__ comb, const float* __restrict__ inj,
                                                           const float* __restrict__ norm, int d, int hc, int T, float* __restrict__ ssq, float* __restrict__ smx, float* __restrict__ part) {
  constexpr int NW = 4 * CS;
  __shared__ __align__(16) uint16_t ah[CS * 32 * 16 * 8];
  __shared__ float wsum[NW][8], wmax[NW][8];
  extern __shared__ __align__(16) float hsum[];          // [2][tiles][4][2][64] (CS == 2)
  const int ks = blockIdx.x, grp = blockIdx.y, tid = threadIdx.x, nks = gridDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = wave & 3, p = wave >> 2, q = lane >> 4;
  const int c0 = ks * 256 * CS, s = c0 / d, i0 = c0 - s * d, K128 = m.cols >> 7, t0 = grp * 8, nt = min(8, T - t0);
  const float nv = norm[(size_t)s * d + i0 + tid];
  // every load the workgroup needs before its first barrier is issued at once: the tokens' weights of the pending update, the streams,
  // the update's vectors (tokens past the end repeat the last one and are dropped), the first row tile's weights
  float v[8], o[8][NP > 0 ? NP : 1];
  const float iv = NP > 0 && tid < 8 ? inj[(t0 + min(tid, nt - 1)) * hc + s] : 0.0f;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int tt = min(t, nt - 1);
    v[t] = x_in[(size_t)(t0 + tt) * in_ts + (size_t)s * in_ss + i0 + tid];
    if constexpr (NP == 1) o[t][0] = comb[(size_t)(t0 + tt) * d + i0 + tid];
    else if constexpr (NP > 1) {
#pragma unroll
      for (int k = 0; k < NP; ++k) o[t][k] = (comb + ((size_t)grp * NP * 8 + tt) * d + i0 + tid)[(size_t)k * 8 * d];
    }
  }
  const int ch0 = ks * 2 * CS + 2 * p;
  WBuf<1> w0, w1; load_w<1>(m, g, ch0, lane, K128, w0); load_w<1>(m, g, ch0 + 1, lane, K128, w1);
  const NibK nk = nib_consts();
  if constexpr (NP > 0) {          // the tokens' weights, once for the workgroup
    if (tid < 8) wmax[0][tid] = 2.0f * b_sigm(iv);
    lds_barrier();
    float wt[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) wt[t] = wmax[0][t];
    lds_barrier();
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      float ov = o[t][0];
#pragma unroll
      for (int k = 1; k < NP; ++k) ov += o[t][k];
      v[t] = v[t] + ov * wt[t];
    }
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = t < nt ? v[t] : 0.0f;
  float xs[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    xs[t] = v[t] * nv;
    if (t < nt) x_out[((size_t)(t0 + t) * hc + s) * d + i0 + tid] = v[t];
    const float ss = wave_sum(v[t] * v[t]), a = wave_max(b_nan_abs(xs[t]));
    if (lane == 0) { wsum[wave][t] = ss; wmax[wave][t] = a; }
  }
  lds_barrier();
  auto slice_max = [&](int t) { float mx = wmax[0][t];
#pragma unroll
    for (int k = 1; k < NW; ++k) mx = fmaxf(mx, wmax[k][t]);
    return mx; };
  if (tid < 8) { float tot = wsum[0][tid];
#pragma unroll
    for (int k = 1; k < NW; ++k) tot += wsum[k][tid];
    ssq[((size_t)grp * nks + ks) * 8 + tid] = tot; smx[((size_t)grp * nks + ks) * 8 + tid] = slice_max(tid); }
#pragma unroll
  for (int t = 0; t < 8; ++t) { float up, dn; b_scale_of(slice_max(t), &up, &dn); uint16_t* o = ah + ((size_t)(tid >> 3) * 16 + 2 * t) * 8 + (tid & 7); b_split(xs[t] * up, o, o + 8); }
  float upf, dn0, dn1; b_scale_of(slice_max(2 * q), &upf, &dn0); b_scale_of(slice_max(2 * q + 1), &upf, &dn1);
  lds_barrier();
  v8h a0[4], a1[4];
#pragma unroll
  for (int st = 0; st < 4; ++st) { a0[st] = __builtin_bit_cast(v8h, ((const uint4*)ah)[(((2 * p) * 4 + st) * 4 + q) * 16 + (lane & 15)]); a1[st] = __builtin_bit_cast(v8h, ((const uint4*)ah)[(((2 * p + 1) * 4 + st) * 4 + q) * 16 + (lane & 15)]); }
  const size_t r64 = (size_t)m.tiles * 64;
  float* pg = part + ((size_t)grp * nks + ks) * 8 * r64;
  for (int tile = 0; tile < m.tiles; ++tile) {
    if (tile * 64 + g * 16 >= m.rows) break;          // (the last tile's padding; nobody reads those rows)
    WDec d0, d1; decode_chunk(w0.w[0], w0.h[0], ch0, nk, d0); decode_chunk(w1.w[0], w1.h[0], ch0 + 1, nk, d1);
    if (tile + 1 < m.tiles) { load_w<1>(m, (tile + 1) * 4 + g, ch0, lane, K128, w0); load_w<1>(m, (tile + 1) * 4 + g, ch0 + 1, lane, K128, w1); }
    v4f c0 = {0.0f, 0.0f, 0.0f, 0.0f}, c1 = c0, tot = c0;
#pragma unroll
    for (int st = 0; st < 4; ++st) { c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0[st], d0.b[st], c0, 0, 0, 0); c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1[st], d1.b[st], c1, 0, 0, 0); }
    scale_add(c0, d0.d, dn0, dn1, tot); scale_add(c1, d1.d, dn0, dn1, tot);
    const float r0 = halves0(tot), r1 = halves1(tot);
    if constexpr (CS == 2) { float* h = hsum + ((((size_t)p * m.tiles + tile) * 4 + g) * 2) * 64 + lane; h[0] = r0; h[64] = r1; }
    else { const size_t row = (size_t)tile * 64 + g * 16 + (lane & 15); pg[(2 * q) * r64 + row] = r0; pg[(2 * q + 1) * r64 + row] = r1; }
  }
  if constexpr (CS == 2) {          // the two chunk pairs' sums meet in shared memory and leave as rows
    lds_barrier();
    for (int i = tid; i < m.tiles * 512; i += 64 * NW) {
      const int tile = i >> 9, t = (i >> 6) & 7, rl = i & 63;
      if (tile * 64 + (rl & 48) >= m.rows) continue;
      const float* h = hsum + (((size_t)tile * 4 + (rl >> 4)) * 2 + (t & 1)) * 64 + (t >> 1) * 16 + (rl & 15);
      pg[t * r64 + tile * 64 + rl] = h[0] + h[(size_t)m.tiles * 512];
    }
  }
}
// ---- second part: grid (8, groups), 256 threads, a workgroup a token: RMS scales, the scaled slice sums, silu -> operand rows ----
// lo: [group][lr / 8][16][8] halves with lo_dn [token]; scl: [token][hc] the streams' RMS scales; opb [token] {up, dn}: the power
// of two of a bound of the token's largest mixed value; inj [token][hc].  At most sixteen slices, lr <= 1024.
__global__ __launch_bounds__(256) void k_blk_mix_lo(const float* __restrict__ part, const float* __restrict__ ssq, const float* __restrict__ smx, int ksplit, int r64, int lr, int hc, int has_inject, float eps, int d, int T,
                                                    uint16_t* __restrict__ lo, float* __restrict__ lo_dn, float* __restrict__ scl, float2* __restrict__ opb, float* __restrict__ inj) {
  __shared__ float sc[16]; __shared__ float bd[4]; __shared__ float wm[4];
  const int t = blockIdx.x, grp = blockIdx.y, ti = grp * 8 + t, tid = threadIdx.x, kps = ksplit / hc, wave = tid >> 6, lane = tid & 63;
  if (ti >= T) return;
  const float* pg = part + ((size_t)grp * ksplit * 8 + t) * r64;
  float pv[16];          // the first round's slices, in flight beside the scales
#pragma unroll
  for (int k = 0; k < 16; ++k) pv[k] = k < ksplit && tid < lr ? pg[(size_t)k * 8 * r64 + tid] : 0.0f;
  float iv[16];
  const bool injt = tid < hc && has_inject;
#pragma unroll
  for (int k = 0; k < 16; ++k) iv[k] = k < ksplit && injt ? pg[(size_t)k * 8 * r64 + lr + tid] : 0.0f;
  if (tid < hc) {
    const float* sp = ssq + ((size_t)grp * ksplit + tid * kps) * 8 + t; const float* mp = smx + ((size_t)grp * ksplit + tid * kps) * 8 + t;
    float tot = sp[0], mx = mp[0];
    for (int k = 1; k < kps; ++k) { tot += sp[k * 8]; mx = fmaxf(mx, mp[k * 8]); }
    const float s = 1.0f / sqrtf(tot / (float)d + eps);
    for (int k = 0; k < kps; ++k) sc[tid * kps + k] = s;
    scl[(size_t)ti * hc + tid] = s; bd[tid] = s * mx;
  }
  lds_barrier();
  auto slice_sum = [&](const float (&v)[16]) { float o = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) if (k < ksplit) { const float tm = v[k] * sc[k]; o = k == 0 ? tm : o + tm; }
    return o; };
  float lv[4]; float mx = 0.0f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    lv[r] = 0.0f;
    if (r * 256 < lr) {
      if (r > 0) {
#pragma unroll
        for (int k = 0; k < 16; ++k) pv[k] = k < ksplit ? pg[(size_t)k * 8 * r64 + r * 256 + tid] : 0.0f;
      }
      const float v = slice_sum(pv) / (float)hc;
      lv[r] = v * b_sigm(v); mx = fmaxf(mx, b_nan_abs(lv[r]));
    }
  }
  mx = wave_max(mx); if (lane == 0) wm[wave] = mx;
  lds_barrier();
  float up, dn; b_scale_of(fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3])), &up, &dn);
  uint16_t* lg = lo + (size_t)grp * lr * 16;
#pragma unroll
  for (int r = 0; r < 4; ++r) if (r * 256 < lr) { const int k = r * 256 + tid; uint16_t* o = lg + ((size_t)(k >> 3) * 16 + 2 * t) * 8 + (k & 7); b_split(lv[r] * up, o, o + 8); }
  if (tid == 0) {
    lo_dn[ti] = dn;
    float b = bd[0]; for (int k = 1; k < hc; ++k) b = fmaxf(b, bd[k]);
    b = b == b ? b : INFINITY;
    float u2, d2; b_scale_of(b, &u2, &d2); opb[ti] = make_float2(u2, d2);
  }
  if (tid < hc) inj[(size_t)ti * hc + tid] = has_inject ? slice_sum(iv) / (float)hc : 0.0f;
}
// ---- third part: up, the gates and the mean of the streams -----------------------------------------------------------------------
// grid (d / 32, cuts of the groups), 2 hc waves: wave (s, g) keeps row group g of the workgroup's 32 rows of stream s of `up`,
// decoded (low rank 256: two chunks, 32 registers), and walks the groups with it; the launch for a window decoded them again
// for every window and redid the whole prologue in each of its workgroups (212 us at 43 windows).  A turn is products, then the
// epilogue's vector instructions, with a barrier between: with 64 columns one workgroup fitted a compute unit and its phases took turns
// (20 us at 301 tokens, 85 at 2000); two of 32 columns overlap theirs, and what a turn reads is asked for a turn ahead (15.9, 70).  Outputs: mixed [token][d] (f32) and, with op and inv given, the same as operand rows.
template <int KC>
__global__ __launch_bounds__(512) void k_blk_mix_up(QMatDev up, const uint4* __restrict__ lo, const float* __restrict__ lo_dn, const float* __restrict__ scl, const float2* __restrict__ opb, const float* __restrict__ x,
                                                     const float* __restrict__ norm, int hc, int d, int T, int per, float* __restrict__ mixed, uint4* __restrict__ op, size_t op_gs, float* __restrict__ inv, int inv_gs) {
  __shared__ __align__(16) uint4 la[2][KC * 256];
  __shared__ float red[4][8][32];
  __shared__ __align__(16) uint16_t st[2][4 * 16 * 8];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4, nw = blockDim.x >> 6;
  const int s = wave >> 1, g = wave & 1, G = (T + 7) >> 3, b0 = blockIdx.y * per, b1 = min(G, b0 + per), col0 = blockIdx.x * 32, nt = blockDim.x >> 5;
  if (b0 >= b1) return;
  WDec wd[KC];
  { const NibK nk = nib_consts(); WBuf<1> w;
#pragma unroll
    for (int c = 0; c < KC; ++c) { load_w<1>(up, ((s * d + col0) >> 4) + g, c, lane, KC, w); decode_chunk(w.w[0], w.h[0], c, nk, wd[c]); } }
  auto fetch = [&](int grp, int buf) { for (int j = wave; j < KC * 4; j += nw) lds_fetch16(lo + (size_t)grp * KC * 256 + j * 64 + lane, &la[buf][j * 64]); };
  // thread = (token, column) of the epilogue; with fewer than 256 threads in rounds
  const int l = tid & 31;
  float nr[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) nr[k] = k < hc ? norm[(size_t)k * d + col0 + l] : 0.0f;
  // what a group's epilogue reads of memory (thread = token tid / 32, column l; the token's factors) and the wave's two tokens' scales
  const int et = tid >> 5;
  float xn[4], sn[4], dn0n, dn1n; float2 obn;
  auto ahead = [&](int grp) {
    const int t0 = grp * 8; const size_t tc = min(t0 + et, T - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) { const bool w = k < hc && et < 8; xn[k] = w ? x[(tc * hc + k) * d + col0 + l] : 0.0f; sn[k] = w ? scl[tc * hc + k] : 0.0f; }
    obn = op && et < 8 ? opb[tc] : make_float2(0.0f, 0.0f);
    dn0n = lo_dn[min(t0 + 2 * q, T - 1)]; dn1n = lo_dn[min(t0 + 2 * q + 1, T - 1)]; };
  fetch(b0, 0); ahead(b0);
  lds_fetch_barrier();
  for (int b = b0; b < b1; ++b) {
    const int buf = (b - b0) & 1, t0 = b * 8;
    const float dn0 = dn0n, dn1 = dn1n; float xv[4], sv[4]; float2 ob = obn;
#pragma unroll
    for (int k = 0; k < 4; ++k) { xv[k] = xn[k]; sv[k] = sn[k]; }
    if (b + 1 < b1) { fetch(b + 1, buf ^ 1); ahead(b + 1); }          // a whole group ahead: a group's own loads would be waited for twice
    __builtin_amdgcn_sched_barrier(0);
    v4f tot = {0.0f, 0.0f, 0.0f, 0.0f};
    { v4f acc[KC];
#pragma unroll
      for (int c = 0; c < KC; ++c) acc[c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < KC; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, la[buf][((c * 4 + j) * 4 + q) * 16 + (lane & 15)]), wd[c].b[j], acc[c], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < KC; ++c) scale_add(acc[c], wd[c].d, dn0, dn1, tot);
    }
    red[s][2 * q][g * 16 + (lane & 15)] = halves0(tot); red[s][2 * q + 1][g * 16 + (lane & 15)] = halves1(tot);
    // the next group's operand and values have arrived behind the products; waiting here and not at the end leaves this group's stores
    // a whole turn to complete
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    for (int t = et; t < 8; t += nt) {
      const int ti = t0 + t; const bool on = ti < T;
      const size_t tc = min(ti, T - 1);
      if (t >= nt) {
#pragma unroll
        for (int k = 0; k < 4; ++k) { xv[k] = k < hc ? x[(tc * hc + k) * d + col0 + l] : 0.0f; sv[k] = k < hc ? scl[tc * hc + k] : 0.0f; }
        if (op) ob = opb[tc];
      }
      float mx = 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) if (k < hc) mx += xv[k] * sv[k] * nr[k] * b_sigm(red[k][t][l]);            // rms: (x * s) * w
      const float mv = mx / (float)hc;
      if (on) mixed[tc * d + col0 + l] = mv;
      if (op) {
        uint16_t* o = st[buf] + ((l >> 3) * 16 + 2 * t) * 8 + (l & 7); b_split(mv * ob.x, o, o + 8);
        if (on && blockIdx.x == 0) for (int sb = l; sb < (d >> 8); sb += 32) inv[(size_t)b * inv_gs + sb * 8 + t] = ob.y;
      }
    }
    lds_barrier();
    if (op && tid < 64) op[(size_t)b * op_gs + (size_t)(col0 >> 3) * 16 + tid] = ((const uint4*)st[buf])[tid];
  }
}

// embedding rows -> one row a token is model.hip's pyre_row_launch; the output of a head of 128 columns as operand rows:
// grid ceil(T * heads * 16 / 256): thread = eight columns; RMS norm of the head's 128 values, gate, the layer's power of two
__global__ __launch_bounds__(256) void k_blk_gdn_out(const float* __restrict__ o, const float* __restrict__ z, int zs, const float* __restrict__ nw, float eps, int heads, int T, float upf, uint4* __restrict__ op, size_t op_gs, float* __restrict__ out) {
  const size_t gi = (size_t)blockIdx.x * 256 + threadIdx.x; const int j = (int)(gi & 15), h = (int)((gi >> 4) % heads); const int ti = (int)((gi >> 4) / heads);
  if (ti >= T) return;
  const float* po = o + ((size_t)ti * heads + h) * 128 + 8 * j; const float* pz = z + (size_t)ti * zs + h * 128 + 8 * j;
  float v[8], zz[8], w[8];
#pragma unroll
  for (int k = 0; k < 8; k += 4) { const float4 a = *(const float4*)(po + k), b = *(const float4*)(pz + k), c = *(const float4*)(nw + 8 * j + k);
    v[k] = a.x; v[k + 1] = a.y; v[k + 2] = a.z; v[k + 3] = a.w; zz[k] = b.x; zz[k + 1] = b.y; zz[k + 2] = b.z; zz[k + 3] = b.w; w[k] = c.x; w[k + 1] = c.y; w[k + 2] = c.z; w[k + 3] = c.w; }
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; ++k) ss += v[k] * v[k];
  ss += wave_dpp<0xB1, 0xf>(0.0f, ss); ss += wave_dpp<0x4E, 0xf>(0.0f, ss); ss += wave_dpp<0x141, 0xf>(0.0f, ss); ss += wave_dpp<0x140, 0xf>(0.0f, ss);          // the head's sixteen lanes
  const float sc = 1.0f / sqrtf(ss / 128.0f + eps);
  float r[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) r[k] = (v[k] * (sc * w[k])) * b_sigm(zz[k]);
  if (out) { float* po2 = out + ((size_t)ti * heads + h) * 128 + 8 * j; *(float4*)po2 = make_float4(r[0], r[1], r[2], r[3]); *(float4*)(po2 + 4) = make_float4(r[4], r[5], r[6], r[7]); }
  if (op) {
    struct H8 { uint16_t v[8]; } a, b;
#pragma unroll
    for (int k = 0; k < 8; ++k) b_split(r[k] * upf, &a.v[k], &b.v[k]);
    uint4* dst = op + (size_t)(ti >> 3) * op_gs + (size_t)(h * 16 + j) * 16 + 2 * (ti & 7);
    dst[0] = __builtin_bit_cast(uint4, a); dst[1] = __builtin_bit_cast(uint4, b);
  }
}

// The same in the per-quarter form of k_gdn_delta_q and its reader load_a_sq (the bits of a window): a quarter of a head, 32 columns,
// is split into halves on its own power of two, brought to the head's largest power by exponent arithmetic, and the head's
// 1 / RMS goes into the chunk's factor, inv + group * inv_gs + head * 8 + token.
__global__ __launch_bounds__(256) void k_blk_gdn_out_q(const float* __restrict__ o, const float* __restrict__ z, int zs, const float* __restrict__ nw, float eps, int heads, int T, uint4* __restrict__ op, size_t op_gs, float* __restrict__ inv, int inv_gs) {
  const size_t gi = (size_t)blockIdx.x * 256 + threadIdx.x; const int j = (int)(gi & 15), h = (int)((gi >> 4) % heads); const int ti = (int)((gi >> 4) / heads);
  if (ti >= T) return;          // (whole rows of sixteen lanes)
  const float* po = o + ((size_t)ti * heads + h) * 128 + 8 * j; const float* pz = z + (size_t)ti * zs + h * 128 + 8 * j;
  float v[8], u[8];
#pragma unroll
  for (int k = 0; k < 8; k += 4) { const float4 a = *(const float4*)(po + k), b = *(const float4*)(pz + k), c = *(const float4*)(nw + 8 * j + k);
    v[k] = a.x; v[k + 1] = a.y; v[k + 2] = a.z; v[k + 3] = a.w;
    u[k] = (a.x * c.x) * b_sigm(b.x); u[k + 1] = (a.y * c.y) * b_sigm(b.y); u[k + 2] = (a.z * c.z) * b_sigm(b.z); u[k + 3] = (a.w * c.w) * b_sigm(b.w); }
  // the order of a wave's sum over the quarter's 32 columns: a tree of neighbours
  float ss = ((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3])) + ((v[4] * v[4] + v[5] * v[5]) + (v[6] * v[6] + v[7] * v[7]));
  ss += wave_dpp<0xB1, 0xf>(0.0f, ss); ss += wave_dpp<0x4E, 0xf>(0.0f, ss);
  float am = b_nan_abs(u[0]);
#pragma unroll
  for (int k = 1; k < 8; ++k) am = fmaxf(am, b_nan_abs(u[k]));
  am = fmaxf(am, wave_dpp<0xB1, 0xf>(0.0f, am)); am = fmaxf(am, wave_dpp<0x4E, 0xf>(0.0f, am));
  float up, dn; b_scale_of(am, &up, &dn);
  float mr = fmaxf(dn, wave_dpp<0x141, 0xf>(0.0f, dn)); mr = fmaxf(mr, wave_dpp<0x140, 0xf>(0.0f, mr));
  const _Float16 f = (_Float16)__uint_as_float(__float_as_uint(dn) - (__float_as_uint(mr) - 0x3F800000u));
  struct H8 { uint16_t v[8]; } a, b;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    b_split(u[k] * up, &a.v[k], &b.v[k]);
    a.v[k] = __builtin_bit_cast(unsigned short, (_Float16)(__builtin_bit_cast(_Float16, a.v[k]) * f)); b.v[k] = __builtin_bit_cast(unsigned short, (_Float16)(__builtin_bit_cast(_Float16, b.v[k]) * f));
  }
  uint4* dst = op + (size_t)(ti >> 3) * op_gs + (size_t)(h * 16 + j) * 16 + 2 * (ti & 7);
  dst[0] = __builtin_bit_cast(uint4, a); dst[1] = __builtin_bit_cast(uint4, b);
  const float q0 = wave_dpp<0x150, 0xf>(0.0f, ss), q1 = wave_dpp<0x154, 0xf>(0.0f, ss), q2 = wave_dpp<0x158, 0xf>(0.0f, ss), q3 = wave_dpp<0x15C, 0xf>(0.0f, ss);
  if (j == 0) inv[(size_t)(ti >> 3) * inv_gs + h * 8 + (ti & 7)] = mr * __builtin_amdgcn_rsqf((((q0 + q1) + q2) + q3) * (1.0f / 128.0f) + eps);
}

// ... and as f32 rows in k_gdn_delta's order: the sum of squares of each half of the head as a tree of neighbours, then the two halves
__global__ __launch_bounds__(256) void k_blk_gdn_out_w(const float* __restrict__ o, const float* __restrict__ z, int zs, const float* __restrict__ nw, float eps, int heads, int T, float* __restrict__ out) {
  const size_t gi = (size_t)blockIdx.x * 256 + threadIdx.x; const int j = (int)(gi & 15), h = (int)((gi >> 4) % heads); const int ti = (int)((gi >> 4) / heads);
  if (ti >= T) return;
  const float* po = o + ((size_t)ti * heads + h) * 128 + 8 * j; const float* pz = z + (size_t)ti * zs + h * 128 + 8 * j; float* pr = out + ((size_t)ti * heads + h) * 128 + 8 * j;
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; k += 4) { const float4 a = *(const float4*)(po + k); v[k] = a.x; v[k + 1] = a.y; v[k + 2] = a.z; v[k + 3] = a.w; }
  float ss = ((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3])) + ((v[4] * v[4] + v[5] * v[5]) + (v[6] * v[6] + v[7] * v[7]));
  ss += wave_dpp<0xB1, 0xf>(0.0f, ss); ss += wave_dpp<0x4E, 0xf>(0.0f, ss); ss += wave_dpp<0x141, 0xf>(0.0f, ss); ss += wave_dpp<0x140, 0xf>(0.0f, ss);
  const float sc = 1.0f / sqrtf(ss / 128.0f + eps);
#pragma unroll
  for (int k = 0; k < 8; ++k) pr[k] = (v[k] * (sc * nw[8 * j + k])) * b_sigm(pz[k]);
}

}  // namespace

// parts: K slices left apart for the mix that follows (PYRE_GEMV_PARTS, as pyre_gemv_parts_launch cuts them), or 1
int pyre_blk_gemm_launch(pyre_ctx* ctx, const QMatDev& m, const uint4* op, size_t op_gs, const float* inv, int inv_gs, int inv_kind, float* y, int ys, int T, int parts) {
  if (m.fmt != FMT_IQ3_S_M || !m.mq || m.cols % 256) return pyre_fail(ctx, PYRE_E_TYPE, "blk_gemm: the matrix is not held in the matrix-core layout");
  int nw, cw; pyre_gemm_m_plan(m, parts, &nw, &cw);
  const int K128 = m.cols / 128, per = (K128 + parts - 1) / parts;
  if (parts > 1) { nw = 4; cw = (per + 3) / 4; }          // (GemvEpi::four_waves)
  if (K128 % parts || nw * cw < per) return pyre_fail(ctx, PYRE_E_SHAPE, "blk_gemm: %d columns in %d slices", m.cols, parts);
  const int G = (T + 7) / 8, bx = (m.tiles + 3) / 4, ish = inv_kind == PYRE_INV_CHUNK ? 0 : 1; const bool uni = inv_kind == PYRE_INV_TOKEN;
  ProfScope ps(ctx, "blk_gemm", qmat_gguf_bytes(m, m.rows) + 4.0 * T * ((double)m.cols + m.rows));
  // Groups a wave meets with a decoded chunk (eight, with running sums to keep four): as few as leave at most a workgroup a compute unit
  // (256), with four K parts, whose workgroups are a quarter as long, two; four until there are 640.  us a launch, 2048 columns:
  // 12352 rows (49 workgroups a group) 32 tokens 21.0 with one, 23.1 with two; 48: 28.0, 23.3; 72: 24.8 with two, 31.3 with four; 104:
  // 33.8, 31.9; 264: 58.5, 46.1; 392: 67.1 with four, 66.9 with eight; 520: 84.2, 70.8; 2048: 258, 228.  9216 rows (36): 72 tokens 28.0
  // with one, 23.6 with two; 136: 32.7 with two, 31.7 with four; 520: 65.6 with four, 66.8 with eight; 776: 85.5, 72.0.  2048 rows of 4096
  // columns in four parts (32): 72 tokens 17.4 with one, 16.4 with two; 200: 21.4 with two, 22.3 with four; 264: 29.9, 27.8.
  const int b2 = bx * parts, tg = b2 * G <= 256 ? 1 : (b2 * ((G + 1) / 2) <= (parts > 1 ? 512 : 256) ? 2 : (cw != 1 || b2 * ((G + 3) / 4) <= 640 ? 4 : 8));
#define BLK_GO(TG, CW1, UNI) hipLaunchKernelGGL((k_blk_gemm<TG, CW1, UNI>), dim3(bx, (G + TG - 1) / TG, parts), dim3(256), (size_t)TG * (per / (ish + 1) + 1) * 8 * 4, ctx->stream, m, op, op_gs, inv, inv_gs, ish, cw, y, ys, T)
  if (cw == 1 && uni) { if (tg == 8) BLK_GO(8, true, true); else if (tg == 4) BLK_GO(4, true, true); else if (tg == 2) BLK_GO(2, true, true); else BLK_GO(1, true, true); }
  else if (cw == 1) { if (tg == 8) BLK_GO(8, true, false); else if (tg == 4) BLK_GO(4, true, false); else if (tg == 2) BLK_GO(2, true, false); else BLK_GO(1, true, false); }
  else { if (tg == 4) BLK_GO(4, false, false); else if (tg == 2) BLK_GO(2, false, false); else BLK_GO(1, false, false); }
#undef BLK_GO
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
int pyre_blk_op_split_launch(pyre_ctx* ctx, const float* x, int cols, int T, uint4* op, size_t op_gs, float* inv, int inv_gs) {
  ProfScope ps(ctx, "blk_op_split", 8.0 * T * cols);
  hipLaunchKernelGGL(k_blk_op_split, dim3(cols / 256, (T + 7) / 8), dim3(256), 0, ctx->stream, x, cols, T, op, op_gs, inv, inv_gs);
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
int pyre_blk_gdn_out_launch(pyre_ctx* ctx, const float* o, const float* z, int zs, const float* nw, float eps, int heads, int T, float up, uint4* op, size_t op_gs, float* out) {
  ProfScope ps(ctx, "blk_gdn_out", 4.0 * T * heads * 128 * 3);
  hipLaunchKernelGGL(k_blk_gdn_out, dim3((unsigned)(((size_t)T * heads * 16 + 255) / 256)), dim3(256), 0, ctx->stream, o, z, zs, nw, eps, heads, T, up, op, op_gs, out);
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}

int pyre_blk_gdn_out_q_launch(pyre_ctx* ctx, const float* o, const float* z, int zs, const float* nw, float eps, int heads, int T, uint4* op, size_t op_gs, float* inv, int inv_gs) {
  ProfScope ps(ctx, "blk_gdn_out", 4.0 * T * heads * 128 * 3);
  hipLaunchKernelGGL(k_blk_gdn_out_q, dim3((unsigned)(((size_t)T * heads * 16 + 255) / 256)), dim3(256), 0, ctx->stream, o, z, zs, nw, eps, heads, T, op, op_gs, inv, inv_gs);
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}

int pyre_blk_gdn_out_w_launch(pyre_ctx* ctx, const float* o, const float* z, int zs, const float* nw, float eps, int heads, int T, float* out) {
  ProfScope ps(ctx, "blk_gdn_out", 4.0 * T * heads * 128 * 3);
  hipLaunchKernelGGL(k_blk_gdn_out_w, dim3((unsigned)(((size_t)T * heads * 16 + 255) / 256)), dim3(256), 0, ctx->stream, o, z, zs, nw, eps, heads, T, out);
  PYRE_CHECK_LAUNCH(ctx); return PYRE_OK;
}
static int blk_mix_cs(const HcDev& h) { return h.d % 512 == 0 ? 2 : 1; }
static int blk_mix_slices(const HcDev& h) { return h.hc * h.d / (256 * blk_mix_cs(h)); }
bool pyre_blk_mix_ok(const HcDev& h) { return pyre_hc_aop_ok(h) && (h.lr == 256 || h.lr == 512) && blk_mix_slices(h) <= 16 && h.d / 256 <= 64; }
size_t pyre_blk_mix_bytes(const HcDev& h, int T) {
  const size_t G = (T + 7) / 8, ks = 16;
  return 8 * 256 + 4 * (2 * G * ks * 8 + G * ks * 8 * ((size_t)h.lr + h.hc + 64) + 8 * G * (1 + h.hc + 2)) + G * h.lr * 32;
}
void pyre_blk_mix_carve(const HcDev& h, int T, void* base, BlkMix* b) {
  uint8_t* p = (uint8_t*)base; auto take = [&](size_t n) { void* r = p; p += (n + 255) & ~(size_t)255; return r; };
  const size_t G = (T + 7) / 8, ks = 16;
  b->ssq = (float*)take(4 * G * ks * 8); b->smx = (float*)take(4 * G * ks * 8); b->part = (float*)take(4 * G * ks * 8 * ((size_t)h.lr + h.hc + 64));
  b->lo = (uint16_t*)take(G * h.lr * 32); b->lo_dn = (float*)take(4 * 8 * G); b->scl = (float*)take(4 * 8 * G * h.hc); b->opb = (float2*)take(8 * 8 * G);
}
// np: vectors of the pending update (0, 1 or PYRE_MOE_GROUPS; see k_blk_mix_down)
int pyre_blk_mix_launch(pyre_ctx* ctx, const HcDev& h, const BlkMix& b, const float* x_in, int in_ss, int in_ts, float* x, int T, const float* comb, int np, const float* comb_inj, float eps,
                        float* mixed, float* inj, uint4* op, size_t op_gs, float* inv, int inv_gs) {
  if (!pyre_blk_mix_ok(h) || (np != 0 && np != 1 && np != PYRE_MOE_GROUPS)) return pyre_fail(ctx, PYRE_E_ARG, "blk_mix: unsupported shape or %d partial vectors", np);
  const int G = (T + 7) / 8, ks = blk_mix_slices(h), cs = blk_mix_cs(h);
  { ProfScope ps(ctx, "blk_mix_down", qmat_gguf_bytes(h.di, h.di.rows) + 4.0 * T * h.hc * h.d * 2);
    const size_t lds = cs == 2 ? (size_t)h.di_m.tiles * 4096 : 0;
#define MIX_GO(NP, CS) hipLaunchKernelGGL((k_blk_mix_down<NP, CS>), dim3(ks, G), dim3(256 * CS), lds, ctx->stream, h.di_m, x_in, in_ss, in_ts, x, comb, comb_inj, h.norm, h.d, h.hc, T, b.ssq, b.smx, b.part)
    if (cs == 2) { if (np == 0) MIX_GO(0, 2); else if (np == 1) MIX_GO(1, 2); else MIX_GO(PYRE_MOE_GROUPS, 2); }
    else { if (np == 0) MIX_GO(0, 1); else if (np == 1) MIX_GO(1, 1); else MIX_GO(PYRE_MOE_GROUPS, 1); }
#undef MIX_GO
  } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "blk_mix_lo", 4.0 * T * ks * h.lr);
    hipLaunchKernelGGL(k_blk_mix_lo, dim3(8, G), dim3(256), 0, ctx->stream, b.part, b.ssq, b.smx, ks, h.di_m.tiles * 64, h.lr, h.hc, h.has_inject ? 1 : 0, eps, h.d, T, b.lo, b.lo_dn, b.scl, b.opb, inj); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "blk_mix_up", qmat_gguf_bytes(h.up, h.up.rows) + 4.0 * T * (h.hc * h.d + 2.0 * h.d));
    const int bx = h.d / 32; int per = (int)std::max<int64_t>(1, (int64_t)bx * G / 1024); per = std::min(per, 16);          // about four workgroups a compute unit, a decoded row group used up to sixteen times
    const dim3 grid(bx, (G + per - 1) / per), blk(h.hc * 128);
    if (h.lr == 256) hipLaunchKernelGGL((k_blk_mix_up<2>), grid, blk, 0, ctx->stream, h.up_m, (const uint4*)b.lo, b.lo_dn, b.scl, b.opb, x, h.norm, h.hc, h.d, T, per, mixed, op, op_gs, inv, inv_gs);
    else hipLaunchKernelGGL((k_blk_mix_up<4>), grid, blk, 0, ctx->stream, h.up_m, (const uint4*)b.lo, b.lo_dn, b.scl, b.opb, x, h.norm, h.hc, h.d, T, per, mixed, op, op_gs, inv, inv_gs); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}
