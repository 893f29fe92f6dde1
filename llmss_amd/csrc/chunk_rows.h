// Infinities and NaN in the chunked forms of the recurrences (linear_scan.hip, delta.hip). A chunk's matrix products multiply a
// token's numbers with zeros for the tokens before it, which is no zero where they are infinite or NaN: unheeded, up to 15 earlier
// tokens would become NaN that a token-by-token walk leaves finite.
#pragma once
#include <float.h>

#include "common.h"

__device__ __forceinline__ double at_least(double x, double lo) { return x < lo ? lo : x; }  // (a NaN stays one, unlike with fmax)

// Takes such numbers of a column out of the products. u: a wave's 16 columns of a chunk's 64 tokens in the accumulator layout (lane (li, g):
// column li, tokens 16 r + 4 g + i). Returns the column's first such token, 64 if there is none; its state is the caller's.
__device__ __forceinline__ int contain(f32x4 (&u)[4], int g) {
  float z = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i) z = fmaf(u[r][i], 0.f, z);
  int bad = 64;
  if (__builtin_expect(__any(z != z), 0)) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!(fabsf(u[r][i]) <= FLT_MAX)) bad = min(bad, 16 * r + 4 * g + i), u[r][i] = 0.f;
    bad = min(bad, __shfl_xor(bad, 16, 64));
    bad = min(bad, __shfl_xor(bad, 32, 64));
  }
  return bad;
}

// The results of sixteen tokens from 16 r on, from here on only added to: what a walk makes of such a number, NaN from its token on
__device__ __forceinline__ void from_bad(f32x4& o, int bad, int r, int g) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (16 * r + 4 * g + i >= bad) o[i] = __uint_as_float(0x7fc00000u);
}

// Both, of four such blocks
__device__ __forceinline__ int contain(f32x4 (&u)[4], f32x4 (&o)[4], int g) {
  const int bad = contain(u, g);
  if (__builtin_expect(__any(bad < 64), 0)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) from_bad(o[r], bad, r, g);
  }
  return bad;
}
