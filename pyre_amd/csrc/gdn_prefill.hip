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

// ---- the recurrence token by token, the bits of k_gdn_delta_q -------------------------------------------------------------------
// A prompt of the model takes this one: its state and outputs are then those of decoding the tokens in windows, to the bit, so
// that no token's expert choice tips with the path the prompt took.  k_gdn_delta_q keeps 32 columns a workgroup, eight rows a
// thread, and adds the sixteen row groups' sums through shared memory behind a barrier: 0.9 us a token.  Here a wave keeps
// four columns, a row of sixteen lanes (a lane: eight rows) each: the sums meet in the same order by DPP row shifts
// (x <- p + x of the lane before, fifteen times: the last lane has ((p0 + p1) + p2) + ..), without a barrier, and the
// output's sums of one token run in the wait slots of the next token's.  About 100 vector instructions a token, one wave a SIMD
// for 32 heads (the recurrence is a chain, so further waves would only share the SIMD).
// grid (nv, 8), 4 waves: workgroup (h, y) columns 16 y .. of head h.  The keys, queries (normalised, co of k_gdnc_conv), values and gate
// inputs of sixteen tokens at a time go through shared memory, the next sixteen in registers meanwhile.
__device__ __forceinline__ float row_shr1(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x111, 0xf, 0xf, true)); }
__device__ __forceinline__ float row_last(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x15F, 0xf, 0xf, true)); }
__global__ __launch_bounds__(256) void k_gdn_rec(GdnDev p, const float* __restrict__ co, const float2* __restrict__ gates, int T, const float* __restrict__ ssm_in, float* __restrict__ ssm_out, float* __restrict__ oraw) {
  constexpr int TB = 16, R = 8;
  __shared__ __align__(16) float4 kq[2][TB][2][2][16];          // [buffer][token][k, q][rows 0-3, 4-7 of a row group][row group]
  __shared__ float vs[2][TB][16], os[2][TB][16]; __shared__ float2 gb[2][TB];
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
  fetch(0); store(0);
  lds_barrier();
  for (int t0 = 0, buf = 0; t0 < T; t0 += TB, buf ^= 1) {
    if (t0 + TB < T) fetch(t0 + TB);
    const int n = min(TB, T - t0);
    // In the wait slots of token t's chain: the output terms of token t - 1 (its state is still there: the decayed one goes to
    // other registers) and the output chain of token t - 2.
    float po2 = 0.0f, po1 = 0.0f; float4 qa = make_float4(0.0f, 0.0f, 0.0f, 0.0f), qb = qa;          // chain input of token t - 2; the query of token t - 1
    auto terms = [&]() { const float q[R] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w}; float o = S[0] * q[0];
#pragma unroll
      for (int r = 1; r < R; ++r) o += S[r] * q[r];
      return o; };
    auto step = [&](const Tok& c, int t) {
      const float k[R] = {c.k0.x, c.k0.y, c.k0.z, c.k0.w, c.k1.x, c.k1.y, c.k1.z, c.k1.w};
      float D[R];
#pragma unroll
      for (int r = 0; r < R; ++r) D[r] = S[r] * c.g.x;
      float pm = D[0] * k[0];
#pragma unroll
      for (int r = 1; r < R; ++r) pm += D[r] * k[r];
      const float q[R] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
      float m = pm, o = po2, pt = S[0] * q[0];
#pragma unroll
      for (int i = 0; i < 15; ++i) {
        m = pm + row_shr1(m); o = po2 + row_shr1(o);
        if (i & 1) { if (i / 2 + 1 < R) pt += S[i / 2 + 1] * q[i / 2 + 1]; }
      }
      if (rg == 15) os[buf][max(t - 2, 0)][jl] = o;          // (the first two tokens' write nothing of use: the next one overwrites it)
      const float delta = (c.v - row_last(m)) * c.g.y;
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = D[r] + k[r] * delta;
      po2 = pt; qa = c.q0; qb = c.q1;
    };
    // a token ahead: the wave is alone on its SIMD, nothing else hides the reads; two sets of registers taking turns
    Tok x0 = get(buf, 0), x1;
    int t = 0;
    for (; t + 1 < n; t += 2) { x1 = get(buf, t + 1); step(x0, t); x0 = get(buf, min(t + 2, n - 1)); step(x1, t + 1); }
    if (t < n) step(x0, t);
    po1 = terms();
    { float o = po2, o1 = po1;
#pragma unroll
      for (int i = 0; i < 15; ++i) { o = po2 + row_shr1(o); o1 = po1 + row_shr1(o1); }
      if (rg == 15) { if (n > 1) os[buf][n - 2][jl] = o; os[buf][n - 1][jl] = o1; } }
    if (t0 + TB < T) store(buf ^ 1);
    lds_barrier();
    if ((tid >> 4) < n) oraw[(size_t)(t0 + (tid >> 4)) * w + (size_t)h * p.dv + cb + (tid & 15)] = os[buf][tid >> 4][tid & 15];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) ssm_out[so + (size_t)r * p.dv] = S[r];
}

// The same for layers in the head-a-workgroup form (k_gdn_delta: four groups of 32 rows a column): a quad of lanes a column, a lane its
// group's 32 rows, the four sums by quad broadcasts in order.  grid (nv, 2), 4 waves: 64 columns a workgroup.
template <int I> __device__ __forceinline__ float quad_lane(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), I * 0x55, 0xf, 0xf, true)); }
__device__ __forceinline__ float quad_sum(float x) { return ((quad_lane<0>(x) + quad_lane<1>(x)) + quad_lane<2>(x)) + quad_lane<3>(x); }
__global__ __launch_bounds__(256) void k_gdn_rec4(GdnDev p, const float* __restrict__ co, const float2* __restrict__ gates, int T, const float* __restrict__ ssm_in, float* __restrict__ ssm_out, float* __restrict__ oraw) {
  constexpr int TB = 8, R = 32;
  __shared__ __align__(16) float ks[2][TB][4][R + 4], qs[2][TB][4][R + 4];          // (a group's row padded: four groups, four banks)
  __shared__ float vs[2][TB][64]; __shared__ float2 gb[2][TB];
  const int h = blockIdx.x, cb = blockIdx.y * 64, kh = h % p.nk, tid = threadIdx.x, lane = tid & 63, g = lane & 3;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), jl = wave * 16 + (lane >> 2);
  const int nqk = p.nk * DK, ch = 2 * nqk + p.nv * p.dv, w = p.nv * p.dv;
  const size_t so = ((size_t)h * DK + g * R) * p.dv + cb + jl;
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) S[r] = ssm_in[so + (size_t)r * p.dv];
  auto load = [&](int t0, int buf) {          // eight tokens: 128 k, 128 q, 64 v each
    for (int i = tid; i < TB * DK; i += 256) { const int t = min(t0 + i / DK, T - 1), c = i % DK; const float* r = co + (size_t)t * ch + kh * DK + c; ks[buf][i / DK][c >> 5][c & 31] = r[nqk]; qs[buf][i / DK][c >> 5][c & 31] = r[0]; }
    for (int i = tid; i < TB * 64; i += 256) vs[buf][i >> 6][i & 63] = co[(size_t)min(t0 + (i >> 6), T - 1) * ch + 2 * nqk + (size_t)h * p.dv + cb + (i & 63)];
    if (tid < TB) gb[buf][tid] = gates[(size_t)min(t0 + tid, T - 1) * p.nv + h];
  };
  load(0, 0);
  lds_barrier();
  for (int t0 = 0, buf = 0; t0 < T; t0 += TB, buf ^= 1) {
    if (t0 + TB < T) load(t0 + TB, buf ^ 1);
    const int n = min(TB, T - t0);
    struct Row { float4 v[8]; };
    auto row = [&](const float* x) { Row r;
#pragma unroll
      for (int i = 0; i < 8; ++i) r.v[i] = *(const float4*)(x + 4 * i);
      return r; };
    Row k = row(ks[buf][0][g]);
    for (int t = 0; t < n; ++t) {          // (the query is read behind the keys' sums, the next token's keys behind the query's)
      const float2 gt = gb[buf][t]; const float vt = vs[buf][t][jl];
      const Row q = row(qs[buf][t][g]);
      const float* kk = (const float*)&k; const float* qq = (const float*)&q;
      float pm = 0.0f;
#pragma unroll
      for (int r = 0; r < R; ++r) { S[r] *= gt.x; pm += S[r] * kk[r]; }
      const float delta = (vt - quad_sum(pm)) * gt.y;
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] += kk[r] * delta;
      k = row(ks[buf][min(t + 1, n - 1)][g]);
      float po = 0.0f;
#pragma unroll
      for (int r = 0; r < R; ++r) po += S[r] * qq[r];
      const float o = quad_sum(po);
      if (g == 0) oraw[(size_t)(t0 + t) * w + (size_t)h * p.dv + cb + jl] = o;
    }
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
    if (!quarters) hipLaunchKernelGGL(k_gdn_rec4, dim3(g.nv, g.dv / 64), dim3(256), 0, ctx->stream, g, b.co, (const float2*)b.dec, T, ssm_in, ssm_out, oraw);
    else hipLaunchKernelGGL(k_gdn_rec, dim3(g.nv, g.dv / 16), dim3(256), 0, ctx->stream, g, b.co, (const float2*)b.dec, T, ssm_in, ssm_out, oraw); } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}
