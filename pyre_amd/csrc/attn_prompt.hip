// Gated attention over the KV cache for a prompt taken layer by layer: hundreds of queries a launch, each with its own view
// (attn_core, dense branch, src/model/qwen4exp_gguf.rs:1558-1615, over the cache of :1519-1534 and src/model/kv4.rs:12-42).
//
// A pass per window of eight tokens reads and converts the cache again for every window and leaves partial sums per chunk of
// 128 positions for a merge: at 8192 tokens 11 000 launches of 19 + 6.5 us.  Here
//   k_att_frag   turns the visible positions once a layer into what the matrix cores read: keys and values as two f16 halves
//                each (v * 2^e = h1 + h2, one power of two per 64 positions and KV head), laid out in the order lanes supply
//                them, so that the pass below only copies
//   k_att_pass   128 rows (query head x token) a workgroup, sixteen a wave: scores, running softmax, weighted values, tile of 32
//                positions by tile, the tiles copied from memory straight into shared memory one ahead
// Positions below a token's packed boundary are read from the 4-bit cache, the others from the f32 planes, as everywhere;
// the boundary moves by 64 every 64 tokens, so the blocks in between are visited in both forms and a token masks the one it
// does not see.  Products of halves are exact, sums f32; the low halves' own product (2^-22 of the term) is left out.
#include "formats.h"
#include <algorithm>

typedef float f4_ __attribute__((ext_vector_type(4)));
typedef _Float16 h8_ __attribute__((ext_vector_type(8)));

namespace {

constexpr int HD = 256, BLK = 64;
constexpr size_t FRAG = 65536;          // bytes of one (block of 64 positions, KV head): keys; the values follow
__device__ __forceinline__ float t_sigm(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ int packed_boundary(const AttnDev& a, int n) { return (a.kv_bits == 4 && n > a.kv_recent + 64) ? ((n - a.kv_recent) / 64) * 64 : 0; }
__device__ __forceinline__ void two_halves(float xs, uint16_t* h1, uint16_t* h2) {
  const _Float16 a = (_Float16)xs, b = (_Float16)(xs - (float)a);
  *h1 = __builtin_bit_cast(unsigned short, a); *h2 = __builtin_bit_cast(unsigned short, b);
}
__device__ __forceinline__ float nibf(uint32_t w, int i) { return (float)(((int)(w << (28 - 4 * i))) >> 28); }

// grid (blocks of 64 positions, nkv), 256 threads: blocks 0 .. npk-1 in packed form, then f32 blocks from fb0.  Output block z = blockIdx.x:
// frag + ((z * nkv + kvh) * 2 FRAG), inverse scales finv[(z * nkv + kvh) * 2 + {0: keys, 1: values}].
//   keys:   [position / 16][dim / 32][half][lane] x 16 B, lane (p, kg): position 16 i + p, dims 32 s + 8 kg .. + 7 in the order 0 4 1 5 2 6 3 7 (the query halves' order)
//   values: [position / 32][dim / 16][half][lane] x 16 B, lane (j, kg): dim 16 i + j, positions 32 s + 8 kg .. + 7
__global__ __launch_bounds__(256) void k_att_frag(AttnDev a, KvDev kv, int npk, int fb0, int n, uint8_t* __restrict__ frag, float* __restrict__ finv) {
  __shared__ float x[BLK][HD + 1]; __shared__ float mx[4];
  const int z = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const bool pk = z < npk; const int b = pk ? z : fb0 + z - npk, p0 = b * BLK; const size_t R = (size_t)a.nkv * HD;
  uint8_t* out = frag + ((size_t)z * a.nkv + kvh) * 2 * FRAG;
  for (int v = 0; v < 2; ++v) {
    __syncthreads();
    float m = 0.0f;
    if (v == 0) {          // keys: position = lane, dims by wave
      const int pos = p0 + lane; const bool on = pos < n;
      if (pk) for (int w = wave; w < HD / 8; w += 4) {
        const uint32_t u = kv.kq[kv_blk((size_t)kvh * (HD / 8) + w, R / 8, pos)]; const float s = kv.ks[kv_blk((size_t)kvh * (HD / 32) + w / 4, R / 32, pos)];
        for (int j = 0; j < 8; ++j) { const float f = nibf(u, j) * s; x[lane][8 * w + j] = f; m = fmaxf(m, fabsf(f)); }
      } else for (int d = wave; d < HD; d += 4) { const float f = on ? kv.kf[kv_blk((size_t)kvh * HD + d, R, pos)] : 0.0f; x[lane][d] = f; const float af = fabsf(f); m = fmaxf(m, af == af ? af : INFINITY); }
    } else {          // values: dim (or word) by thread
      if (pk) for (int i = tid; i < BLK * (HD / 8); i += 256) {
        const int p = i >> 5, w = i & 31; const uint32_t u = kv.vq[(size_t)(p0 + p) * (R / 8) + (size_t)kvh * (HD / 8) + w]; const float s = kv.vs[(size_t)(p0 + p) * (R / 32) + (size_t)kvh * (HD / 32) + w / 4];
        for (int j = 0; j < 8; ++j) { const float f = nibf(u, j) * s; x[p][8 * w + j] = f; m = fmaxf(m, fabsf(f)); }
      } else for (int p = 0; p < BLK; ++p) { const float f = p0 + p < n ? kv.vf[(size_t)(p0 + p) * R + (size_t)kvh * HD + tid] : 0.0f; x[p][tid] = f; const float af = fabsf(f); m = fmaxf(m, af == af ? af : INFINITY); }
    }
    m = wave_max(m); if (lane == 0) mx[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
    int e = 0;
    if (m > 0.0f && m < INFINITY) { e = 140 - (int)((__float_as_uint(m) >> 23) & 0xFF); e = e > 100 ? 100 : e; }
    const float up = __uint_as_float((uint32_t)(127 + e) << 23);
    if (tid == 0) finv[((size_t)z * a.nkv + kvh) * 2 + v] = __uint_as_float((uint32_t)(127 - e) << 23);
    uint4* o = (uint4*)(out + (size_t)v * FRAG);
    for (int i = tid; i < 2048; i += 256) {          // a lane's eight numbers, both halves
      const int ln = i & 63, r = ln & 15, kg = ln >> 4, f = i >> 6; struct H8 { uint16_t h[8]; } a1, a2;
      for (int j = 0; j < 8; ++j) {
        float val;
        if (v == 0) { const int dj = (j & 1) * 4 + (j >> 1); val = x[16 * (f >> 3) + r][32 * (f & 7) + 8 * kg + dj]; }
        else val = x[32 * (f >> 4) + 8 * kg + j][16 * (f & 15) + r];
        two_halves(val * up, &a1.h[j], &a2.h[j]);
      }
      o[(size_t)f * 128 + ln] = __builtin_bit_cast(uint4, a1); o[(size_t)f * 128 + 64 + ln] = __builtin_bit_cast(uint4, a2);
    }
  }
}

template <int CTRL> __device__ __forceinline__ float dpp(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xf, 0xf, false)); }
__device__ __forceinline__ float max16(float v) { v = fmaxf(v, dpp<0xB1>(v)); v = fmaxf(v, dpp<0x4E>(v)); v = fmaxf(v, dpp<0x141>(v)); return fmaxf(v, dpp<0x140>(v)); }
__device__ __forceinline__ float sum16(float v) { v += dpp<0xB1>(v); v += dpp<0x4E>(v); v += dpp<0x141>(v); return v + dpp<0x140>(v); }

// grid (tiles of 128 / G tokens, nkv), 8 waves; the last tiles, with the longest views, first.  qh [token][head][2][256], qsc [token][head]
// (k_attn_prep); out [token][head * 256] = softmax(q K^T / sqrt(hd)) V * sigmoid(gate), the gate beside the query in qkv.
// Shared memory: two tiles of 32 positions, 64 KB each (keys and values, both halves), and the softmax weights' halves a wave.
// Per tile a wave runs 96 matrix instructions (1536 clocks, two waves a SIMD); its fragments are 64 KB of shared-memory reads,
// 512 KB a workgroup and tile = 4096 clocks: the shared memory sets the pace, about 1.7 us a tile.
template <int G>
__global__ __launch_bounds__(512, 2) void k_att_pass(AttnDev a, const uint16_t* __restrict__ qh, const float* __restrict__ qsc, const float* __restrict__ qkv, int stride, int start, int T, int npk, int fb0,
                                                     const uint8_t* __restrict__ frag, const float* __restrict__ finv, float* __restrict__ out) {
  extern __shared__ __align__(16) uint8_t sm[];
  uint4* kvs = (uint4*)sm;                                // [2][keys 2048 | values 2048]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, q = lane >> 4;
  uint16_t* ps = (uint16_t*)(sm + 131072) + wave * 2 * 16 * 40;          // [half][row][32 + 8]
  constexpr int TT = 128 / G;
  const int tile = (int)gridDim.x - 1 - (int)blockIdx.x, kvh = blockIdx.y, tk0 = tile * TT, tk1 = min(T, tk0 + TT);
  const int ra = 16 * wave + r, ta = min(tk0 + ra / G, T - 1), ha = kvh * G + ra % G;          // the row whose query this lane supplies
  h8_ q1[8], q2[8];
  { const uint16_t* p = qh + ((size_t)ta * a.nh + ha) * 2 * HD + 8 * q;
#pragma unroll
    for (int s = 0; s < 8; ++s) { q1[s] = __builtin_bit_cast(h8_, *(const uint4*)(p + 32 * s)); q2[s] = __builtin_bit_cast(h8_, *(const uint4*)(p + HD + 32 * s)); } }
  int pos[4], pb[4]; float qs[4];          // the four rows whose sums this lane holds
#pragma unroll
  for (int e = 0; e < 4; ++e) { const int row = 16 * wave + 4 * q + e, t = min(tk0 + row / G, T - 1); pos[e] = start + t; pb[e] = packed_boundary(a, pos[e] + 1); qs[e] = qsc[(size_t)t * a.nh + kvh * G + row % G] * 0.0625f; }
  static_assert(HD == 256, "1 / sqrt(hd)");
  // tiles: packed blocks below the last token's boundary, then f32 blocks from the first token's boundary to the last token
  const int pk1 = packed_boundary(a, start + tk1) / BLK, f0 = packed_boundary(a, start + tk0 + 1) / BLK, ntp = 2 * pk1, nt = ntp + (start + tk1 - f0 * BLK + 31) / 32;
  auto src = [&](int i) -> size_t { const int z = i < ntp ? i >> 1 : npk + f0 - fb0 + ((i - ntp) >> 1); return (size_t)z * a.nkv + kvh; };
  auto fetch = [&](int i, int buf) {
    const int hb = i < ntp ? i & 1 : (i - ntp) & 1; const uint8_t* b = frag + src(i) * 2 * FRAG + (size_t)hb * (FRAG / 2);
#pragma unroll
    for (int j = 0; j < 8; ++j) { const int o = wave * 8 + j; const uint8_t* g = b + (o >= 32 ? FRAG : 0) + (size_t)(o & 31) * 1024 + lane * 16;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g, (__attribute__((address_space(3))) void*)(kvs + (size_t)buf * 4096 + o * 64), 16, 0, 0); }
  };
  f4_ O[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) O[i] = f4_{0.0f, 0.0f, 0.0f, 0.0f};
  float m[4], l[4], vrun = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) { m[e] = -INFINITY; l[e] = 0.0f; }
  fetch(0, 0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");          // (the fetches a wave issued have landed)
  for (int i = 0; i < nt; ++i) {
    const int buf = i & 1; if (i + 1 < nt) fetch(i + 1, buf ^ 1);
    const bool pk = i < ntp; const int k0 = pk ? i * 32 : f0 * BLK + (i - ntp) * 32;
    const float kinv = finv[src(i) * 2], vinv = finv[src(i) * 2 + 1];
    const uint4* kb = kvs + (size_t)buf * 4096; const uint4* vb = kb + 2048;
    f4_ S[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f4_ acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const h8_ k1 = __builtin_bit_cast(h8_, kb[((j * 8 + s) * 2) * 64 + lane]), k2 = __builtin_bit_cast(h8_, kb[((j * 8 + s) * 2 + 1) * 64 + lane]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(q1[s], k1, acc, 0, 0, 0); acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(q1[s], k2, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(q2[s], k1, acc, 0, 0, 0);
      }
      S[j] = acc;
    }
    // the values' power of two: O is kept in the largest unit met so far
    if (vinv > vrun) {
      if (vrun > 0.0f) { const float f = vrun / vinv;
#pragma unroll
        for (int d = 0; d < 16; ++d) O[d] *= f; }
      vrun = vinv;
    }
    const float pf = 8192.0f * (vinv / vrun);
    float sc[4]; bool moved = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float s[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) { const int key = k0 + 16 * j + r; const bool on = pk ? key < pb[e] : (key >= pb[e] && key <= pos[e]); s[j] = on ? S[j][e] * (qs[e] * kinv) : -INFINITY; }
      const float mn = fmaxf(m[e], max16(fmaxf(s[0], s[1])));
      sc[e] = mn == -INFINITY ? 1.0f : expf(m[e] - mn); moved |= sc[e] != 1.0f; m[e] = mn;
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float p = s[j] == -INFINITY ? 0.0f : expf(s[j] - mn); sum += p;
        uint16_t* o = ps + (4 * q + e) * 40 + 16 * j + r; two_halves(p * pf, o, o + 16 * 40);
      }
      l[e] = l[e] * sc[e] + sum;
    }
    if (__ballot(moved)) {
#pragma unroll
      for (int d = 0; d < 16; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) O[d][e] *= sc[e];
    }
    // (the wave's own shared memory: its operations execute in order)
    __builtin_amdgcn_wave_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const h8_ p1 = __builtin_bit_cast(h8_, *(const uint4*)(ps + r * 40 + 8 * q)), p2 = __builtin_bit_cast(h8_, *(const uint4*)(ps + 16 * 40 + r * 40 + 8 * q));
#pragma unroll
    for (int d = 0; d < 16; ++d) {
      const h8_ v1 = __builtin_bit_cast(h8_, vb[(d * 2) * 64 + lane]), v2 = __builtin_bit_cast(h8_, vb[(d * 2 + 1) * 64 + lane]);
      O[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p1, v1, O[d], 0, 0, 0); O[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p1, v2, O[d], 0, 0, 0);
      O[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p2, v1, O[d], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");          // (the fetches a wave issued have landed)
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = 16 * wave + 4 * q + e, t = tk0 + row / G, h = kvh * G + row % G;
    const float L = sum16(l[e]);
    if (t < tk1) {
      const float f = vrun * (1.0f / 8192.0f); const float* gate = qkv + (size_t)t * stride + (size_t)h * 2 * HD + HD + r; float* o = out + ((size_t)t * a.nh + h) * HD + r;
#pragma unroll
      for (int d = 0; d < 16; ++d) o[16 * d] = (O[d][e] * f / L) * t_sigm(gate[16 * d]);
    }
  }
}

}  // namespace

// blocks the two forms need for queries start .. start + T - 1: npk packed ones from position 0, f32 ones from fb0
static void att_blocks(const AttnDev& a, int start, int T, int* npk, int* fb0, int* nf) {
  *npk = (int)(pyre_packed_boundary((size_t)start + T, a.kv_bits, a.kv_recent) / BLK); *fb0 = (int)(pyre_packed_boundary((size_t)start + 1, a.kv_bits, a.kv_recent) / BLK);
  *nf = (start + T + BLK - 1) / BLK - *fb0;
}
size_t pyre_attn_prompt_bytes(const AttnDev& a, int start, int T) {
  int npk, fb0, nf; att_blocks(a, start, T, &npk, &fb0, &nf);
  return (size_t)(npk + nf) * a.nkv * (2 * FRAG + 8) + 512;
}
int pyre_attn_prompt_launch(pyre_ctx* ctx, const AttnDev& a, const KvDev& kv, const uint16_t* qh, const float* qsc, const float* qkv, int stride, int start, int T, void* scratch, float* out) {
  const int G = a.nh / a.nkv;
  if (a.hd != HD || (G != 1 && G != 2 && G != 4 && G != 8)) return pyre_fail(ctx, PYRE_E_SHAPE, "attention prompt: head dim %d, group size %d unsupported", a.hd, G);
  if (T < 1 || start < 0 || start + T > kv.cap) return pyre_fail(ctx, PYRE_E_STATE, "attention prompt: positions %d..%d outside the cache (%d)", start, start + T, kv.cap);
  int npk, fb0, nf; att_blocks(a, start, T, &npk, &fb0, &nf);
  uint8_t* frag = (uint8_t*)scratch; float* finv = (float*)(frag + (size_t)(npk + nf) * a.nkv * 2 * FRAG);
  { ProfScope ps(ctx, "attn_prompt_frag", (double)(npk + nf) * a.nkv * 2 * FRAG);
    hipLaunchKernelGGL(k_att_frag, dim3(npk + nf, a.nkv), dim3(256), 0, ctx->stream, a, kv, npk, fb0, start + T, frag, finv); } PYRE_CHECK_LAUNCH(ctx);
  { ProfScope ps(ctx, "attn_prompt_pass", (double)(npk + nf) * a.nkv * 2 * FRAG);
    const size_t lds = 131072 + 8 * 2 * 16 * 40 * 2; const int TT = 128 / G;
#define ATT_GO(GG) do { static const hipError_t once = hipFuncSetAttribute((const void*)k_att_pass<GG>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); (void)once; \
      hipLaunchKernelGGL((k_att_pass<GG>), dim3((T + TT - 1) / TT, a.nkv), dim3(512), lds, ctx->stream, a, qh, qsc, qkv, stride, start, T, npk, fb0, frag, finv, out); } while (0)
    if (G == 8) ATT_GO(8); else if (G == 4) ATT_GO(4); else if (G == 2) ATT_GO(2); else ATT_GO(1);
#undef ATT_GO
  } PYRE_CHECK_LAUNCH(ctx);
  return PYRE_OK;
}
