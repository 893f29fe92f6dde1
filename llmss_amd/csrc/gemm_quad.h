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

bool gemm_quad_ok(int N, int K, int64_t ldx, int64_t ldw, int64_t rows, const void* Y, int64_t ldy, int es, bool glu);
void launch_gemm_quad(int grp, const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, const bf16_t* bias, bf16_t* Y,
                      int64_t ldy, int M, int N, int K, int act, int glu, int group_m, unsigned nwg, const PpGroup& gr,
                      hipStream_t st, const QkvEpi* qe = nullptr);
