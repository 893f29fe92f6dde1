// Element access for kernels that run in either bf16 or fp32 storage (math is fp32 in both).
//
// The kernels of the fp32-residual block (resid32.hip), the strided / grouped GEMMs (gemm_any.hip, moe.hip) and
// the latent attention (attention_latent.hip) are templates over the storage type: bf16_t serves a model in its
// serving precision, float runs the same code as a true 32-bit model (no reduced-precision matrix mode).
#pragma once
#include "common.h"

template <typename T>
struct El;

template <>
struct El<float> {
  static __device__ __forceinline__ float ld(const float* p) { return *p; }
  static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
};

template <>
struct El<bf16_t> {
  static __device__ __forceinline__ float ld(const bf16_t* p) { return bf2f(*p); }
  static __device__ __forceinline__ void st(bf16_t* p, float v) { *p = f2bf(v); }
};

// Four neighbouring numbers of a row, at a multiple of four
template <typename T>
__device__ __forceinline__ f32x4 ld4(const T* p) {
  if constexpr (sizeof(T) == 4) return *reinterpret_cast<const f32x4*>(p);
  const u16x4 q = *reinterpret_cast<const u16x4*>(p);
  return f32x4{bf2f(q[0]), bf2f(q[1]), bf2f(q[2]), bf2f(q[3])};
}
template <typename T>
__device__ __forceinline__ void st4(T* p, f32x4 v) {
  if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4*>(p) = v;
  else *reinterpret_cast<u16x4*>(p) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
}

// Four columns (V f32x4) or one (float) of a product whose K was split: the sum of `slabs` fp32 slabs `stride` apart, eight loads in flight,
// added in their order
template <typename V>
__device__ __forceinline__ V slab_sum(const float* p, int slabs, int64_t stride) {
  const V zero = {};
  V a = zero;
  for (int s0 = 0; s0 < slabs; s0 += 8) {
    V v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const V*>(p + min(s0 + j, slabs - 1) * stride);
#pragma unroll
    for (int j = 0; j < 8; ++j) a += s0 + j < slabs ? v[j] : zero;
  }
  return a;
}

// x as the sum of three bf16 numbers (cut off, not rounded: 8 bits each, 24 together, nothing left over), into place j of each
__device__ __forceinline__ void split3(float x, int j, s16x8& h, s16x8& m, s16x8& l) {
  const float a = __uint_as_float(__float_as_uint(x) & 0xffff0000u), y = x - a;
  const float b = __uint_as_float(__float_as_uint(y) & 0xffff0000u), z = y - b;
  h[j] = (short)(__float_as_uint(a) >> 16);
  m[j] = (short)(__float_as_uint(b) >> 16);
  l[j] = (short)(__float_as_uint(z) >> 16);
}

// dtype codes shared with the Python launchers: 0 = bf16, 1 = fp32
#define DISPATCH_T(code, T, ...)                    \
  do {                                              \
    if ((code) == 0) {                              \
      typedef bf16_t T;                             \
      __VA_ARGS__;                                  \
    } else if ((code) == 1) {                       \
      typedef float T;                              \
      __VA_ARGS__;                                  \
    } else {                                        \
      throw std::runtime_error("bad dtype code");   \
    }                                               \
  } while (0)
