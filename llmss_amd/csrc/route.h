// Routing of one token by a group of lanes: what the routers of moe.hip and the closing op of sandwich.hip share.
#pragma once
#include "common.h"

// L lanes route one token of up to L * J outputs: lane e holds the logits of e (and e + 64; bias added; -inf past the last) and what
// corr adds to their scores; an output's rank among all choice values (ties: the lower index first) says whether and where it is
// chosen. row: LDS, 16-byte aligned, room for the outputs in whole fours. (The reads of the row unrolled, groups of lanes no wider than the
// outputs: with two outputs a lane and a wave a token whatever their number, this was a third of a prompt's routing.)
template <int L, int J>
__device__ __forceinline__ void route_ranked(float (&sc)[J], const float (&cr)[J], float* row, int* __restrict__ idx,
                                             float* __restrict__ wts, int E, int top, int norm, int smax) {
  static_assert(L == 64 || J == 1, "several outputs a lane: whole waves");
  const int lane = threadIdx.x & (L - 1);
  auto all_max = [](float x) {
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
    return x;
  };
  auto all_sum = [](float x) {
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
  };
  float ch[J];
  float mx = -INFINITY, den = 0.f;
  if (smax) {
#pragma unroll
    for (int j = 0; j < J; ++j) mx = fmaxf(mx, sc[j]);
    mx = all_max(mx);
  }
  if (smax == 1) {
#pragma unroll
    for (int j = 0; j < J; ++j) den += lane + 64 * j < E ? expf(sc[j] - mx) : 0.f;
    den = all_sum(den);
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int e = lane + 64 * j;
    if (smax != 2 && e < E) sc[j] = smax ? expf(sc[j] - mx) / den : 1.f / (1.f + expf(-sc[j]));
    ch[j] = e < E ? sc[j] + cr[j] : -INFINITY;
    if (!(ch[j] == ch[j])) ch[j] = -INFINITY;  // (a NaN ranks last: the ranks stay a permutation)
    if (e < ((E + 3) & ~3)) row[e] = ch[j];
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  int rank[J];
#pragma unroll
  for (int j = 0; j < J; ++j) rank[j] = 0;
#pragma unroll 4
  for (int e0 = 0; e0 < E; e0 += 4) {  // (the last four are filled up with -inf behind every output: they count for none)
    const f32x4 o = *reinterpret_cast<const f32x4*>(row + e0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) rank[j] += o[i] > ch[j] || (o[i] == ch[j] && e0 + i < lane + 64 * j) ? 1 : 0;
  }
  float sum = 0.f;
  bool in[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    in[j] = lane + 64 * j < E && rank[j] < top;
    if (smax == 2) sc[j] = expf(sc[j] - mx);  // (the largest is always chosen)
    sum += in[j] ? sc[j] : 0.f;
  }
  sum = all_sum(sum);
  const float inv = smax == 2 ? 1.f / sum : norm ? 1.f / (sum + 1e-20f) : 1.f;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (in[j]) {
      idx[rank[j]] = lane + 64 * j;
      wts[rank[j]] = sc[j] * inv;
    }
}

// the same by a whole wave, what corr adds to outputs `lane` and `lane` + 64 in cr
__device__ __forceinline__ void route_ranked(float (&sc)[2], float* row, const float (&cr)[2], int* __restrict__ idx,
                                             float* __restrict__ wts, int E, int top, int norm, int smax) {
  if (E > 64) {
    route_ranked<64, 2>(sc, cr, row, idx, wts, E, top, norm, smax);
  } else {
    float s1[1] = {sc[0]};
    const float c1[1] = {cr[0]};
    route_ranked<64, 1>(s1, c1, row, idx, wts, E, top, norm, smax);
  }
}

// the same, corr in memory or null
__device__ __forceinline__ void route_ranked(float (&sc)[2], float* row, const float* __restrict__ corr, int* __restrict__ idx,
                                             float* __restrict__ wts, int E, int top, int norm, int smax) {
  const int lane = threadIdx.x & 63;
  float cr[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) cr[j] = corr && lane + 64 * j < E ? corr[lane + 64 * j] : 0.f;
  route_ranked(sc, row, cr, idx, wts, E, top, norm, smax);
}
