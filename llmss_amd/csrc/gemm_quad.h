// What the 256 x 256 prompt GEMMs (gemm.hip's ping-pong kernel and gemm_quad.hip) share.
#pragma once
#include "common.h"

struct PpGroup {  // grouped expert products: the tile list of moe.hip
  const int* meta = nullptr;
  const int* order = nullptr;
  int E = 0, maxt = 0, top = 1;
  int64_t sB = 0;       // elements between the experts' weights
  float* Yf = nullptr;  // GRP 2
  // GRP 3: gate weights beside the up weights, the pairs' weights (null: 1) and the activation's parameters
  const bf16_t* Wu = nullptr;
  const float* pw = nullptr;
  float limit = 0.f, alpha = 0.f;
  int silu = 0;
};

// silu(g) u, or the clamped form
__device__ __forceinline__ float glu_clamped_t(float g, float u, float limit, float alpha, int silu) {
  if (silu) return g / (1.f + expf(-g)) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + 1.f);
}

// g / (1 + exp(-alpha z)), for 128 numbers a lane at the end of a tile: exp2 of a product held in two numbers (k + kl is -alpha log2(e)) and a
// quotient by the hardware's reciprocal, one unit of its last place off, together up to 3.2e-7 before the result is rounded to bf16 (g / (1 +
// expf()) 3.6e-7; numbers under 1e-36 may come out as zero; products of 1024 x 4096 x 2048 with either gate are off their 64-bit value by the
// same 0.0016605 with both). Half of that one's instructions: with expf the gates of a tile took 8.7 us of 66. 8192 x 8192 x 2048 with its gate
// 214 -> 197 us, 8192 x 22016 x 4096 1017 -> 987.
// An infinite z leaves the product's rest no number, which is cut, so that infinities and NaN come out as they do there.
__device__ __forceinline__ float gate_by(float g, float z, float k, float kl) {
  const float t = z * k, r = __builtin_amdgcn_fmed3f(fmaf(z, kl, fmaf(z, k, -t)), -1.f, 1.f);
  const float e = __builtin_amdgcn_exp2f(t) * fmaf(r, 0.6931471805599453f, 1.f);
  return g * __builtin_amdgcn_rcpf(1.f + e);
}
constexpr double kLog2e = 1.4426950408889634, kGeluTwice = 1.5957691216057308;  // (GELU: 2 sqrt(2 / pi))
__device__ __forceinline__ float silu_gate_by(float g) { return gate_by(g, g, (float)-kLog2e, (float)((double)(float)kLog2e - kLog2e)); }
__device__ __forceinline__ float gelu_gate_by(float g) {
  constexpr double k = kGeluTwice * kLog2e;
  return gate_by(g, g + 0.044715f * g * g * g, (float)-k, (float)((double)(float)k - k));
}

// glu_clamped_t with that gate and without a branch: SiLU is the clamped form with limits that are not numbers (the minimum of x and NaN is x),
// alpha 1 and nothing added.
struct GluForm {
  float limit, k, kl, add;
  __device__ __forceinline__ GluForm(float lim, float alpha, int silu) {
    const double f = -kLog2e * (silu ? 1.0 : (double)alpha);
    k = (float)f;
    kl = (float)(f - (double)k);
    limit = silu ? __builtin_nanf("") : lim;
    add = silu ? 0.f : 1.f;
  }
  __device__ __forceinline__ float operator()(float g, float u) const {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit) + add;
    return gate_by(g, g, k, kl) * u;
  }
};

bool gemm_quad_ok(int N, int K, int64_t ldx, int64_t ldw, int64_t rows, const void* Y, int64_t ldy, int es, bool glu,
                  bool list = false);
void launch_gemm_quad(int grp, const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, const bf16_t* bias, bf16_t* Y,
                      int64_t ldy, int M, int N, int K, int act, int glu, int group_m, unsigned nwg, const PpGroup& gr,
                      hipStream_t st, const QkvEpi* qe = nullptr);
