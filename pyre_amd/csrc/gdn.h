// The delta rule's sums over a head's 128 rows, in the one order that every kernel of the recurrence keeps (gdn.hip for a step
// and a window, gdn_prefill.hip for a prompt), so that a token's bits are the same in all of them: eight rows a group as two
// chains of four, the sixteen groups as a tree of neighbours.  A column's sum is the recurrence's serial chain: nine dependent
// operations here, against twenty-two with the groups added one after the other (rows in one chain of eight, then fifteen adds).
//   mem = g sum_r S_r k_r,  delta = (v - mem) beta,  S_r = g S_r + k_r delta,  o = sum_r S_r q_r       (linear_core, :1655-1668)
#pragma once
#include "common.h"
#ifdef __HIPCC__
__device__ __forceinline__ float gdn_dot8(const float* S, const float* k) {
  float a = S[0] * k[0], b = S[4] * k[4];
#pragma unroll
  for (int r = 1; r < 4; ++r) { a = fmaf(S[r], k[r], a); b = fmaf(S[4 + r], k[4 + r], b); }
  return a + b;
}
// N group sums, N a power of two: neighbours first
template <int N> __device__ __forceinline__ float gdn_tree(const float (&p)[N]) {
  float v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = p[i];
#pragma unroll
  for (int s = 1; s < N; s *= 2)
#pragma unroll
    for (int i = 0; i + s < N; i += 2 * s) v[i] += v[i + s];
  return v[0];
}
// the sum of a lane of the wave's lower half and its counterpart in the upper half, in both
__device__ __forceinline__ float halves_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
#endif
