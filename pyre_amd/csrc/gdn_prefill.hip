// Gated DeltaNet over a prompt in chunked form on the fp32 matrix cores (v_mfma_f32_16x16x4_f32).
//
// The reference has no chunked form (linear_core runs the recurrence token by token, src/model/qwen4exp_gguf.rs:
// 1654-1670); this is the same recurrence regrouped per chunk of C = 64 tokens.  With L_i = sum_{j<=i} log g_j inside
// the chunk and S_0 the state at its start,
//     (I + A) Delta = diag(beta) (V - diag(e^L) K S_0),   A_ij = beta_i e^{L_i-L_j} k_i.k_j  (j < i)
//     o_i     = e^{L_i} S_0^T q_i + sum_{j<=i} P_ij delta_j,   P_ij = e^{L_i-L_j} q_i.k_j
//     S_C     = e^{L_C} S_0 + sum_j e^{L_C-L_j} k_j (x) delta_j
// Every decay factor is the exponential of a non-positive difference of log-decays, so nothing overflows however
// strong the gate is.  Delta is linear in S_0:  Delta = U - W S_0 with (I + A) [W | U] = [diag(beta e^L) K | diag(beta) V], so
// everything but three products with the state is done for all chunks at once:
//   k_gdnc_conv   convolution, SiLU, L2 norms, k once more transposed                     (all tokens)
//   k_gdnc_chunk  A, P, the solve for W and U                                             (chunks x heads workgroups)
//   k_gdnc_scan   Delta, the outputs and the state, chunk after chunk                     (heads x 8 workgroups of 16 state columns)
// When one workgroup did all of it per chunk a chunk took 39 us and a prompt of 4096 tokens 2.5 ms (the serial solve, with half of
// the chip idle); the scan, now the only serial part, is three small products.  fp32 throughout.
// Tokens past T in the last chunk have beta = 0, k = q = 0 and no decay: they leave the state as it is.
#include "formats.h"

typedef float v4f_ __attribute__((ext_vector_type(4)));

namespace {

constexpr int C = 64, DK = 128;
__device__ __forceinline__ float p_sigm(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float p_softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }
// four steps of a 16x16x4 product: lane (row, q) holds a[i] = A[row][4 q + i], b[i] = B[4 q + i][column]: the sum over sixteen k
__device__ __forceinline__ v4f_ mac16(const float4& a, const float4& b, v4f_ acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0); acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0); return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
}
__device__ __forceinline__ float4 as4(const v4f_& v) { return make_float4(v[0], v[1], v[2], v[3]); }

// grid (ch / 256, ceil(Tp / 16)), 256 threads: thread = channel, sixteen tokens (the taps and the history are fetched once for
// them).  Channels of q and k: two heads a workgroup, L2-normalised over their 128 channels (q also x 1/sqrt(dk)); k also goes to kt
// [chunk][key head][128][64].  Tokens T .. Tp-1 (the last chunk's padding) become zeros.
template <int KK>
__global__ __launch_bounds__(256) void k_gdnc_conv(GdnDev p, const float* __restrict__ proj, int stride, int T, int Tp, const float* __restrict__ conv_in, float* __restrict__ conv_out, float* __restrict__ co, float* __restrict__ kt, float2* __restrict__ gates) {
  __shared__ float red[4][16];
  const int c = blockIdx.x * 256 + threadIdx.x, t0 = blockIdx.y * 16, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int nqk = p.nk * DK, ch = 2 * nqk + p.nv * p.dv; const bool in = c < ch;
  if (gates && (int)blockIdx.x == (ch + 255) / 256) {          // one more workgroup a group of tokens: decay and beta of every head, gates [token][head]
    for (int i = tid; i < 16 * p.nv; i += 256) { const int t = t0 + i / p.nv, h = i % p.nv; if (t < T) { const float* pr = proj + (size_t)t * stride + ch + p.nv * p.dv; gates[(size_t)t * p.nv + h] = make_float2(expf(p_softplus(pr[p.nv + h] + p.dt[h]) * p.a[h]), p_sigm(pr[h])); } }
    return;
  }
  const int kk = KK ? KK : p.conv_k;
  float w[8], h[16 + 7];          // h[7 + i]: token t0 + i; before it the history
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = in && k < kk ? p.conv_w[(size_t)c * kk + k] : 0.0f;
#pragma unroll
  for (int i = 0; i < 16 + 7; ++i) {
    const int t = t0 + i - 7; h[i] = 0.0f;
    if (in && t < T && i >= 7 - (kk - 1)) h[i] = t >= 0 ? proj[(size_t)t * stride + c] : (t >= -(kk - 1) ? conv_in[(size_t)(kk - 1 + t) * ch + c] : 0.0f);
  }
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float o = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) if (k == kk - 1) o = w[k] * h[7 + i];
#pragma unroll
    for (int k = 0; k < 7; ++k) if (k < kk - 1) {          // tap k reads token i - (kk - 1) + k
      float hv = 0.0f;
#pragma unroll
      for (int b = 0; b < 8; ++b) if (b == kk - 1 - k) hv = h[7 + i - b];
      o += w[k] * hv;
    }
    v[i] = t0 + i < T ? o * p_sigm(o) : 0.0f;
  }
  if (blockIdx.x * 256 < 2 * nqk) {          // (uniform: 2 nk heads of 128 channels, two a workgroup; nk even or the last pair ends with a head of v, whose factor stays 1)
#pragma unroll
    for (int i = 0; i < 16; ++i) { const float s = wave_sum(v[i] * v[i]); if (lane == 0) red[wave][i] = s; }
    lds_barrier();
    if (c < 2 * nqk) {
      const float f = c < nqk ? 1.0f / sqrtf((float)DK) : 1.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = v[i] * ((1.0f / sqrtf(red[wave & 2][i] + red[(wave & 2) + 1][i] + 1e-6f)) * f);
    }
  }
  if (!in) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) co[(size_t)(t0 + i) * ch + c] = v[i];
  if (kt && c >= nqk && c < 2 * nqk) {
    float* k2 = kt + (((size_t)(t0 / C) * p.nk + (c - nqk) / DK) * DK + (c - nqk) % DK) * C + t0 % C;
#pragma unroll
    for (int i = 0; i < 16; i += 4) *(float4*)(k2 + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
  }
  if (t0 <= T - 1 && T - 1 < t0 + 16) for (int k = 0; k < kk - 1; ++k) {          // (the last group of sixteen writes conv_out, the first reads conv_in, in no order: never the same buffer)
    const int src = T - (kk - 1) + k;
    if (src >= 0) conv_out[(size_t)k * ch + c] = proj[(size_t)src * stride + c];
    else { float hv = 0.0f;
#pragma unroll
      for (int i = 0; i < 7; ++i) if (i - 7 == src) hv = h[i];
      conv_out[(size_t)k * ch + c] = hv; }
  }
}

// grid (chunks, nv), 4 waves.  dec [chunk][head][2][64]: e^{L_i}, e^{L_C-L_j}.
__global__ __launch_bounds__(256) void k_gdnc_chunk(GdnDev p, const float* __restrict__ co, const float* __restrict__ proj, int stride, int T, float* __restrict__ W, float* __restrict__ U, float* __restrict__ P, float* __restrict__ dec) {
  __shared__ __align__(16) float Ks[C][DK + 4], Qs[C][DK + 4], A[C][C + 4], Ti[4][16][20];          // (rows padded against bank conflicts); A holds -A below its diagonal blocks, A inside them
  __shared__ double L[C]; __shared__ float Bt[C], eL[C];
  const int ck = blockIdx.x, h = blockIdx.y, kh = h % p.nk, tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nqk = p.nk * DK, ch = 2 * nqk + p.nv * p.dv, w = p.nv * p.dv, t0 = ck * C;
  const float* qc = co + (size_t)t0 * ch + (size_t)kh * DK; const float* kc = qc + nqk; const float* vc = co + (size_t)t0 * ch + 2 * nqk + (size_t)h * p.dv;
  for (int i = tid; i < C * (DK / 4); i += 256) { const int row = i >> 5, c4 = (i & 31) * 4; *(float4*)&Ks[row][c4] = *(const float4*)(kc + (size_t)row * ch + c4); *(float4*)&Qs[row][c4] = *(const float4*)(qc + (size_t)row * ch + c4); }
  if (wave == 0) {
    const bool on = t0 + lane < T; const float* pr = proj + (size_t)(on ? t0 + lane : 0) * stride + ch + w;
    float lg = on ? p_softplus(pr[p.nv + h] + p.dt[h]) * p.a[h] : 0.0f; const float bt = on ? p_sigm(pr[h]) : 0.0f;
    // the running sum in double: with strong gates it reaches thousands inside a chunk, and what counts are differences of
    // neighbours' sums, which in f32 would keep three digits
    double run = 0.0, mine = 0.0;
#pragma unroll
    for (int i = 0; i < C; ++i) { run += (double)__int_as_float(__builtin_amdgcn_readlane(__float_as_int(lg), i)); if (lane == i) mine = run; }
    L[lane] = mine; Bt[lane] = bt; const float e = expf((float)mine); eL[lane] = e;
    float* d = dec + ((size_t)ck * p.nv + h) * 2 * C; d[lane] = e; d[C + lane] = expf((float)(run - mine));
  }
  __syncthreads();
  // A and P: ten 16x16 tiles on or below the diagonal each, five a wave
#pragma unroll
  for (int u = 0; u < 5; ++u) {
    const int job = wave * 5 + u, which = job >= 10 ? 1 : 0, ix = job - 10 * which, ti = ix >= 6 ? 3 : (ix >= 3 ? 2 : (ix >= 1 ? 1 : 0)), tj = ix - ti * (ti + 1) / 2;
    const float* ar = which ? &Qs[16 * ti + r][4 * q] : &Ks[16 * ti + r][4 * q]; const float* br = &Ks[16 * tj + r][4 * q];
    v4f_ acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k0 = 0; k0 < DK; k0 += 16) acc = mac16(*(const float4*)(ar + k0), *(const float4*)(br + k0), acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 16 * ti + 4 * q + e, j = 16 * tj + r; const float dc = j <= i ? expf((float)(L[i] - L[j])) : 0.0f;
      if (which) P[(((size_t)ck * p.nv + h) * C + i) * C + j] = dc * acc[e];
      else { const float a = j < i ? Bt[i] * dc * acc[e] : 0.0f; A[i][j] = ti == tj ? a : -a; }
    }
  }
  __syncthreads();
  // the diagonal blocks' inverses, a wave each, a column a lane: x_i = delta_ic - sum_{k<i} A_ik x_k
  if (lane < 16) {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s = i == lane ? 1.0f : 0.0f;
#pragma unroll
      for (int k = 0; k < 16; ++k) if (k < i) s = fmaf(-A[16 * wave + i][16 * wave + k], x[k], s);
      x[i] = s; Ti[wave][i][lane] = s;
    }
  }
  __syncthreads();
  // W and U by block rows: D_i = T_ii (B_i - sum_{k<i} A_ik D_k); a wave four column tiles of [W | U] at a time
#pragma unroll 1
  for (int u = 0; u < 4; ++u) {
    const int ct = 4 * wave + u, col = (ct & 7) * 16 + r; const bool is_w = ct < 8;
    v4f_ D[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v4f_ acc;
#pragma unroll
      for (int e = 0; e < 4; ++e) { const int row = 16 * i + 4 * q + e; acc[e] = is_w ? Bt[row] * eL[row] * Ks[row][col] : Bt[row] * vc[(size_t)row * ch + col]; }
#pragma unroll
      for (int k = 0; k < 4; ++k) if (k < i) acc = mac16(*(const float4*)&A[16 * i + r][16 * k + 4 * q], as4(D[k]), acc);
      const v4f_ z = {0.0f, 0.0f, 0.0f, 0.0f};
      D[i] = mac16(*(const float4*)&Ti[i][r][4 * q], as4(acc), z);
      float* o = (is_w ? W : U) + (((size_t)ck * p.nv + h) * C + 16 * i + 4 * q) * DK + col;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[(size_t)e * DK] = D[i][e];
    }
  }
}

// grid (nv, dv / 16), 4 waves: sixteen columns of a head's state through all chunks.  The state lies in shared memory transposed, so
// that four consecutive rows of a column -- what a lane supplies to four steps of the product and receives from it -- are one
// 16-byte access.  Per chunk: W S_0 and Q S_0 (a row tile a wave) | P Delta, S update (two row tiles a wave).
__global__ __launch_bounds__(256) void k_gdnc_scan(GdnDev p, const float* __restrict__ co, const float* __restrict__ kt, const float* __restrict__ W, const float* __restrict__ U, const float* __restrict__ P, const float* __restrict__ dec,
                                                   int nch, int T, const float* __restrict__ ssm_in, float* __restrict__ ssm_out, float* __restrict__ oraw) {
  __shared__ __align__(16) float St[16][DK + 4], Dt[16][C + 4], Dd[16][C + 4];          // S, Delta, Delta x e^{L_C-L_j}: [column][row]
  const int h = blockIdx.x, cb = blockIdx.y * 16, kh = h % p.nk, tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nqk = p.nk * DK, ch = 2 * nqk + p.nv * p.dv, w = p.nv * p.dv;
  const float* sin_ = ssm_in + (size_t)h * DK * p.dv + cb; float* sout = ssm_out + (size_t)h * DK * p.dv + cb;
  for (int i = tid; i < DK * 16; i += 256) St[i & 15][i >> 4] = sin_[(size_t)(i >> 4) * p.dv + (i & 15)];
  float4 wf[8], qf[8]; float uf[4];
  auto fetch = [&](int c) {
    const float* wr = W + (((size_t)c * p.nv + h) * C + 16 * wave + r) * DK + 4 * q; const float* qr = co + (size_t)(c * C + 16 * wave + r) * ch + (size_t)kh * DK + 4 * q;
#pragma unroll
    for (int k = 0; k < 8; ++k) { wf[k] = *(const float4*)(wr + 16 * k); qf[k] = *(const float4*)(qr + 16 * k); }
    const float* ur = U + (((size_t)c * p.nv + h) * C + 16 * wave + 4 * q) * DK + cb + r;
#pragma unroll
    for (int e = 0; e < 4; ++e) uf[e] = ur[(size_t)e * DK];
  };
  fetch(0);
  __syncthreads();
  for (int c = 0; c < nch; ++c) {
    const float* pr = P + (((size_t)c * p.nv + h) * C + 16 * wave + r) * C + 4 * q; const float* kr = kt + (((size_t)c * p.nk + kh) * DK + 32 * wave + r) * C + 4 * q; const float* dc = dec + ((size_t)c * p.nv + h) * 2 * C;
    float4 pf[4], kf[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { pf[j] = j <= wave ? *(const float4*)(pr + 16 * j) : make_float4(0.0f, 0.0f, 0.0f, 0.0f); kf[0][j] = *(const float4*)(kr + 16 * j); kf[1][j] = *(const float4*)(kr + 16 * C + 16 * j); }
    const float4 e1 = *(const float4*)(dc + 16 * wave + 4 * q), e2 = *(const float4*)(dc + C + 16 * wave + 4 * q); const float eC = dc[C - 1];
    v4f_ aw = {0.0f, 0.0f, 0.0f, 0.0f}, aq = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 8; ++k) { const float4 s = *(const float4*)&St[r][16 * k + 4 * q]; aw = mac16(wf[k], s, aw); aq = mac16(qf[k], s, aq); }
    float4 d; d.x = uf[0] - aw[0]; d.y = uf[1] - aw[1]; d.z = uf[2] - aw[2]; d.w = uf[3] - aw[3];
    *(float4*)&Dt[r][16 * wave + 4 * q] = d;
    *(float4*)&Dd[r][16 * wave + 4 * q] = make_float4(d.x * e2.x, d.y * e2.y, d.z * e2.z, d.w * e2.w);
    aq[0] *= e1.x; aq[1] *= e1.y; aq[2] *= e1.z; aq[3] *= e1.w;
    lds_barrier();
    if (c + 1 < nch) fetch(c + 1);
#pragma unroll
    for (int u = 0; u < 2; ++u) {          // the state first: the next chunk waits for it
      float4* sp = (float4*)&St[r][32 * wave + 16 * u + 4 * q]; const float4 s = *sp;
      v4f_ a = {eC * s.x, eC * s.y, eC * s.z, eC * s.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) a = mac16(kf[u][j], *(const float4*)&Dd[r][16 * j + 4 * q], a);
      *sp = as4(a);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) if (j <= wave) aq = mac16(pf[j], *(const float4*)&Dt[r][16 * j + 4 * q], aq);
    const int ti = c * C + 16 * wave + 4 * q;
#pragma unroll
    for (int e = 0; e < 4; ++e) if (ti + e < T) oraw[(size_t)(ti + e) * w + (size_t)h * p.dv + cb + r] = aq[e];
    lds_barrier();
  }
  for (int i = tid; i < DK * 16; i += 256) sout[(size_t)(i >> 4) * p.dv + (i & 15)] = St[i & 15][i >> 4];
}

// ---- the recurrence token by token, the bits of the step and window kernels -------------------------------------------------------
// A prompt of the model takes this one: its state and outputs are then those of decoding the tokens in windows, to the bit, so
// that no token's expert choice tips with the path the prompt took.  The step kernels add their row groups' sums through shared
// memory behind a barrier: 0.9 us a token.  Here a wave keeps four columns, a row of sixteen lanes (a lane: eight rows) each, and the sums
// meet in the step kernels' order without a barrier: one lane after the other's sum is an operand of the add, read by a row shift, so
// that the running sum itself never passes through a shift (a value that was just written can be shifted only two instructions later:
// x <- p + x of the lane before, fifteen times, took three slots a step).  The output's row-group sums go to the wave's own shared memory and are
// added sixteen tokens at a time, a lane an output.  About 80 vector instructions a token, one wave a SIMD for 32 heads (the recurrence is a
// chain, so further waves would only share the SIMD).  2048 tokens of the A3B layer: both chains by shifts of the running sum 574 us, the output's through
// shared memory and the sum unshifted 481, moves apart from the adds 421; 200 tokens of the other form 160 -> 81.
// QUARTERS: k_gdn_delta_q's sums, sixteen groups of eight rows; else k_gdn_delta's, four groups of 32 rows (a quad of lanes), whose
// output is summed on the spot.
// grid (nv, 8), 4 waves: workgroup (h, y) columns 16 y .. of head h.  The keys, queries (normalised, co of k_gdnc_conv), values and gate
// inputs of sixteen tokens at a time go through shared memory, the next sixteen in registers meanwhile.
template <int CTRL> __device__ __forceinline__ float dpp(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true)); }
// ... as a move of its own: folded into the add that uses it, the running sum would be an operand of a shifting instruction, two slots after its last
template <int CTRL> __device__ __forceinline__ float dpp_mov(float x) { float v = dpp<CTRL>(x); asm("" : "+v"(v)); return v; }
// lane 15 of a row: ((p of lane 0 + p of lane 1) + p of lane 2) + ..
__device__ __forceinline__ float row_chain16(float p) {
  const float v[15] = {dpp_mov<0x11F>(p), dpp_mov<0x11E>(p), dpp_mov<0x11D>(p), dpp_mov<0x11C>(p), dpp_mov<0x11B>(p), dpp_mov<0x11A>(p), dpp_mov<0x119>(p), dpp_mov<0x118>(p),
                       dpp_mov<0x117>(p), dpp_mov<0x116>(p), dpp_mov<0x115>(p), dpp_mov<0x114>(p), dpp_mov<0x113>(p), dpp_mov<0x112>(p), dpp_mov<0x111>(p)};
  float x = v[0];
#pragma unroll
  for (int i = 1; i < 15; ++i) x += v[i];
  return x + p;
}
template <int L> __device__ __forceinline__ void quad_add8(const float (&p)[8], float& x) {          // x += lane L of the quad's eight, in order
#pragma unroll
  for (int r = 0; r < 8; ++r) { const float v = dpp_mov<L * 0x55>(p[r]); x = (L == 0 && r == 0) ? v : x + v; }
}
// lane 15 of a row: four quads' sums of 32 products in order, added in order
__device__ __forceinline__ float row_chain32(const float (&p)[8]) {
  float x = 0.0f; quad_add8<0>(p, x); quad_add8<1>(p, x); quad_add8<2>(p, x); quad_add8<3>(p, x);
  return ((dpp_mov<0x11C>(x) + dpp_mov<0x118>(x)) + dpp_mov<0x114>(x)) + x;
}
template <bool QUARTERS>
__global__ __launch_bounds__(256) void k_gdn_rec(GdnDev p, const float* __restrict__ co, const float2* __restrict__ gates, int T, const float* __restrict__ ssm_in, float* __restrict__ ssm_out, float* __restrict__ oraw) {
  constexpr int TB = 16, R = 8, OP = 20;
  __shared__ __align__(16) float4 kq[2][TB][2][2][16];          // [buffer][token][k, q][rows 0-3, 4-7 of a row group][row group]
  __shared__ float vs[2][TB][16]; __shared__ float2 gb[2][TB];
  // the wave's output terms: [token][column][row group], or of four tokens [token][column][row] (in steps of 36: a row group's 32)
  __shared__ __align__(16) float po[4][QUARTERS ? TB * 4 * OP : 4 * 4 * 4 * 36];
  const int h = blockIdx.x, cb = blockIdx.y * 16, kh = h % p.nk, tid = threadIdx.x, lane = tid & 63, rg = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), jl = wave * 4 + (lane >> 4), col = cb + jl;
  const int nqk = p.nk * DK, ch = 2 * nqk + p.nv * p.dv, w = p.nv * p.dv;
  const size_t so = ((size_t)h * DK + rg * R) * p.dv + col;
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) S[r] = ssm_in[so + (size_t)r * p.dv];
  float4 f0, f1, f2, f3; float fv; float2 fg = make_float2(0.0f, 0.0f);
  auto src = [&](int t0, int i) { const int e = tid + 256 * i, t = min(t0 + (e >> 6), T - 1), f = e & 63; return *(const float4*)(co + (size_t)t * ch + (f < 32 ? nqk : 0) + kh * DK + 4 * (f & 31)); };
  auto fetch = [&](int t0) {          // token t0 + e / 64's float4 e % 64: 32 of k, 32 of q (past the end: the last token's again)
    f0 = src(t0, 0); f1 = src(t0, 1); f2 = src(t0, 2); f3 = src(t0, 3);
    fv = co[(size_t)min(t0 + (tid >> 4), T - 1) * ch + 2 * nqk + (size_t)h * p.dv + cb + (tid & 15)];
    if (tid < TB) fg = gates[(size_t)min(t0 + tid, T - 1) * p.nv + h];
  };
  auto put = [&](int buf, int i, const float4& f) { const int e = tid + 256 * i, c = e & 63; kq[buf][e >> 6][c >> 5][c & 1][(c & 31) >> 1] = f; };
  auto store = [&](int buf) {
    put(buf, 0, f0); put(buf, 1, f1); put(buf, 2, f2); put(buf, 3, f3);
    vs[buf][tid >> 4][tid & 15] = fv;
    if (tid < TB) gb[buf][tid] = fg;
  };
  struct Tok { float4 k0, k1, q0, q1; float2 g; float v; };
  auto get = [&](int buf, int t) { return Tok{kq[buf][t][0][0][rg], kq[buf][t][0][1][rg], kq[buf][t][1][0][rg], kq[buf][t][1][1][rg], gb[buf][t], vs[buf][t][jl]}; };
  auto step = [&](const Tok& c) {
    const float k[R] = {c.k0.x, c.k0.y, c.k0.z, c.k0.w, c.k1.x, c.k1.y, c.k1.z, c.k1.w}; float m;
#pragma unroll
    for (int r = 0; r < R; ++r) S[r] *= c.g.x;
    if constexpr (QUARTERS) {
      float pm = S[0] * k[0];
#pragma unroll
      for (int r = 1; r < R; ++r) pm += S[r] * k[r];
      m = row_chain16(pm);
    } else {
      float pr[R];
#pragma unroll
      for (int r = 0; r < R; ++r) pr[r] = S[r] * k[r];
      m = row_chain32(pr);
    }
    const float delta = (c.v - dpp<0x15F>(m)) * c.g.y;          // (lane 15's)
#pragma unroll
    for (int r = 0; r < R; ++r) S[r] += k[r] * delta;
  };
  auto out = [&](const Tok& c, int t) {
    const float q[R] = {c.q0.x, c.q0.y, c.q0.z, c.q0.w, c.q1.x, c.q1.y, c.q1.z, c.q1.w};
    if constexpr (QUARTERS) {
      float o = S[0] * q[0];
#pragma unroll
      for (int r = 1; r < R; ++r) o += S[r] * q[r];
      po[wave][(t * 4 + (lane >> 4)) * OP + rg] = o;
    } else {
      float4* d = (float4*)&po[wave][(((t & 3) * 4 + (lane >> 4)) * 4 + (rg >> 2)) * 36 + (rg & 3) * 8];
      d[0] = make_float4(S[0] * q[0], S[1] * q[1], S[2] * q[2], S[3] * q[3]); d[1] = make_float4(S[4] * q[4], S[5] * q[5], S[6] * q[6], S[7] * q[7]);
    }
  };
  // four tokens' outputs from their products: lane = (token, column, row group), then the groups in order
  auto out4 = [&](int t) {
    __builtin_amdgcn_wave_barrier();
    const float4* s = (const float4*)&po[wave][lane * 36]; float x = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) { const float4 v = s[i]; x = i == 0 ? v.x : x + v.x; x += v.y; x += v.z; x += v.w; }
    const float o = ((dpp_mov<0x00>(x) + dpp_mov<0x55>(x)) + dpp_mov<0xAA>(x)) + dpp_mov<0xFF>(x);
    const int ti = t + (lane >> 4);
    if ((lane & 3) == 0 && ti < T) oraw[(size_t)ti * w + (size_t)h * p.dv + cb + wave * 4 + ((lane >> 2) & 3)] = o;
    __builtin_amdgcn_wave_barrier();
  };
  fetch(0); store(0);
  lds_barrier();
  for (int t0 = 0, buf = 0; t0 < T; t0 += TB, buf ^= 1) {
    if (t0 + TB < T) fetch(t0 + TB);
    const int n = min(TB, T - t0);
    if (n == TB) {          // a token ahead: the wave is alone on its SIMD, nothing else hides the reads; two sets of registers taking turns
      Tok x[2]; x[0] = get(buf, 0);
#pragma unroll
      for (int t = 0; t < TB; ++t) { if (t + 1 < TB) x[(t + 1) & 1] = get(buf, t + 1); step(x[t & 1]); out(x[t & 1], t); if (!QUARTERS && (t & 3) == 3) out4(t0 + t - 3); }
    } else for (int t = 0; t < n; ++t) { const Tok x = get(buf, t); step(x); out(x, t); if (!QUARTERS && ((t & 3) == 3 || t + 1 == n)) out4(t0 + (t & ~3)); }
    if constexpr (QUARTERS) {          // lane = (token to, column c of the wave's four)
      __builtin_amdgcn_wave_barrier();
      const int to = lane >> 2, c = lane & 3;
      if (to < n) {
        const float4* s = (const float4*)&po[wave][(to * 4 + c) * OP]; const float4 a = s[0], b = s[1], d = s[2], e = s[3];
        oraw[(size_t)(t0 + to) * w + (size_t)h * p.dv + cb + wave * 4 + c] = ((((((((((((((a.x + a.y) + a.z) + a.w) + b.x) + b.y) + b.z) + b.w) + d.x) + d.y) + d.z) + d.w) + e.x) + e.y) + e.z) + e.w;
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (t0 + TB < T) store(buf ^ 1);
    lds_barrier();
  }
#pragma unroll
  for (int r = 0; r < R; ++r) ssm_out[so + (size_t)r * p.dv] = S[r];
}

}  // namespace

size_t pyre_gdn_chunk_bytes(const GdnDev& g, int T) {
  const size_t nch = ((size_t)T + C - 1) / C, ch = 2 * (size_t)g.nk * g.dk + (size_t)g.nv * g.dv;
  return 6 * 256 + 4 * (nch * C * ch + nch * g.nk * DK * C + nch * g.nv * (2 * (size_t)C * DK + (size_t)C * C + 2 * C));
}
void pyre_gdn_chunk_carve(const GdnDev& g, int T, void* base, GdnChunk* b) {
  const size_t nch = ((size_t)T + C - 1) / C, ch = 2 * (size_t)g.nk * g.dk + (size_t)g.nv * g.dv;
  uint8_t* p = (uint8_t*)base; auto take = [&](size_t n) { void* r = p; p += (n * 4 + 255) & ~(size_t)255; return (float*)r; };
  b->co = take(nch * C * ch); b->kt = take(nch * g.nk * DK * C); b->w = take(nch * g.nv * C * DK); b->u = take(nch * g.nv * C * DK); b->p = take(nch * g.nv * C * C); b->dec = take(nch * g.nv * 2 * C);
}
int pyre_gdn_chunk_launch(pyre_ctx* ctx, const GdnDev& g, const GdnChunk& b, const float* proj, int stride, int T, const float* conv_in, float* conv_out, const float* ssm_in, float* ssm_out, float* oraw) {
  if (g.dk != 128 || g.dv != 128) return pyre_fail(ctx, PYRE_E_SHAPE, "gdn prompt: head dims %dx%d unsupported (128x128 only)", g.dk, g.dv);
  if (T < 1 || g.conv_k < 1 || g.conv_k > 8 || conv_in == conv_out) return pyre_fail(ctx, PYRE_E_ARG, "gdn prompt: %d tokens, %d taps%s", T, g.conv_k, conv_in == conv_out ? ", the history in place" : "");
  const int ch = 2 * g.nk * g.dk + g.nv * g.dv, nch = (T + C - 1) / C, Tp = nch * C;
  { ProfScope ps(ctx, "gdn_prompt_conv", 8.0 * T * ch);
    if (g.conv_k == 4) hipLaunchKernelGGL(k_gdnc_conv<4>, dim3((ch + 255) / 256, Tp / 16), dim3(256), 0, ctx->stream, g, proj, stride, T, Tp, conv_in, conv_out, b.co, b.kt, (float2*)nullptr);
    else hipLaunchKernelGGL(k_gdnc_conv<0>, dim3((ch + 255) / 256, Tp / 16), dim3(256), 0, ctx->stream, g, proj, stride, T, Tp, conv_in, conv_out, b.co, b.kt, (float2*)nullptr); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "gdn_prompt_chunk", 4.0 * T * (ch + g.nv * (2.0 * DK + C)));
    hipLaunchKernelGGL(k_gdnc_chunk, dim3(nch, g.nv), dim3(256), 0, ctx->stream, g, b.co, proj, stride, T, b.w, b.u, b.p, b.dec); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "gdn_prompt_scan", 8.0 * g.nv * g.dk * g.dv + 4.0 * T * g.nv * (4.0 * DK + C));
    hipLaunchKernelGGL(k_gdnc_scan, dim3(g.nv, g.dv / 16), dim3(256), 0, ctx->stream, g, b.co, b.kt, b.w, b.u, b.p, b.dec, nch, T, ssm_in, ssm_out, oraw); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}

// the same steps with the recurrence token by token, bit for bit that of the windows' kernels (pyre_gdn_launch with GdnQ); ssm_in == ssm_out is fine, conv_in == conv_out is not
int pyre_gdn_rec_launch(pyre_ctx* ctx, const GdnDev& g, const GdnChunk& b, const float* proj, int stride, int T, const float* conv_in, float* conv_out, const float* ssm_in, float* ssm_out, float* oraw, bool quarters) {
  if (g.dk != 128 || g.dv != 128) return pyre_fail(ctx, PYRE_E_SHAPE, "gdn prompt: head dims %dx%d unsupported (128x128 only)", g.dk, g.dv);
  if (T < 1 || g.conv_k < 1 || g.conv_k > 8 || conv_in == conv_out) return pyre_fail(ctx, PYRE_E_ARG, "gdn prompt: %d tokens, %d taps%s", T, g.conv_k, conv_in == conv_out ? ", the history in place" : "");
  const int ch = 2 * g.nk * g.dk + g.nv * g.dv, Tp = (T + 15) / 16 * 16;
  { ProfScope ps(ctx, "gdn_prompt_conv", 8.0 * T * ch);
    if (g.conv_k == 4) hipLaunchKernelGGL(k_gdnc_conv<4>, dim3((ch + 255) / 256 + 1, Tp / 16), dim3(256), 0, ctx->stream, g, proj, stride, T, Tp, conv_in, conv_out, b.co, (float*)nullptr, (float2*)b.dec);
    else hipLaunchKernelGGL(k_gdnc_conv<0>, dim3((ch + 255) / 256 + 1, Tp / 16), dim3(256), 0, ctx->stream, g, proj, stride, T, Tp, conv_in, conv_out, b.co, (float*)nullptr, (float2*)b.dec); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "gdn_prompt_rec", 8.0 * g.nv * g.dk * g.dv + 4.0 * T * (ch + 2.0 * g.nv * g.dv));
    if (!quarters) hipLaunchKernelGGL(k_gdn_rec<false>, dim3(g.nv, g.dv / 16), dim3(256), 0, ctx->stream, g, b.co, (const float2*)b.dec, T, ssm_in, ssm_out, oraw);
    else hipLaunchKernelGGL(k_gdn_rec<true>, dim3(g.nv, g.dv / 16), dim3(256), 0, ctx->stream, g, b.co, (const float2*)b.dec, T, ssm_in, ssm_out, oraw); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}
