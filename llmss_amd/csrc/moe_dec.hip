// Grouped expert products of a few rows per expert (decode steps; bf16), over moe.hip's tile list with 16 rows per tile.
//
// Bound by the experts' weights, each read once: a step of 33 tokens over 32 experts of 2048 x 768 reads 300 MB. A workgroup takes two
// groups of 16 weight rows - 16 gate and their 16 up rows, or 32 rows of one matrix - against a tile's 16 rows; its four waves
// split K and meet in LDS, and a wave asks for eight steps of 32 at once (24 KB in flight a wave) straight into the matrix
// instructions' operands: no staging, no barrier before the end, two steps to a 128-byte line. The 64-row tiles that larger steps
// take keep one step of 64 in flight and four waves behind barriers.
// All products of a layer, weights from memory, against those (us): 32 experts of 2048 x 768, 4 rows each, 81 -> 75; 16 of 1024 x 512
// 37 -> 25; 8 of 4096 x 2048 120 -> 86, one row each 110 -> 63. A tile more for an expert reads its weights again.
#include "anytype.h"
#include "gemm_quad.h"

enum { MD_GLU = 0, MD_GELU = 1, MD_DOWN = 2 };

struct MoeDecArgs {
  const bf16_t* X;
  int64_t ldx;
  const bf16_t* W;   // gate (MD_GLU), up (MD_GELU) or down
  const bf16_t* W2;  // MD_GLU: up; null: gate and up rows of W in alternating groups of 16
  void* C;           // [pairs, N]: bf16, MD_DOWN fp32
  int N, K;
  const int* meta;
  const int* order;
  const float* pw;   // weights on the inputs, or null
  int E, maxt, top, silu;
  float limit, alpha;
};

template <int MODE>
__global__ __launch_bounds__(256, 4) void moe_dec_kernel(MoeDecArgs p) {
  constexpr int U = 8;
  __shared__ __attribute__((aligned(16))) float part[4][2][16][20];  // (rows of 20: 16-byte places, spread over the banks)
  if ((int)blockIdx.y >= p.meta[0]) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, g = lane >> 4, K = p.K;
  const int e = p.meta[1 + (p.E + 1) + blockIdx.y], row0 = p.meta[1 + (p.E + 1) + p.maxt + blockIdx.y];
  const int rows = min(16, p.meta[1 + e + 1] - row0);
  const int n0 = blockIdx.x * (MODE == MD_GLU ? 16 : 32);
  const int xr = row0 + min(li, rows - 1);
  const bf16_t* x = p.X + (int64_t)(MODE == MD_DOWN ? xr : p.order[xr] / p.top) * p.ldx + 8 * g;
  const bf16_t *wa, *wb;
  if constexpr (MODE == MD_GLU) {
    const int n = min(n0 + li, p.N - 1);
    if (p.W2) {
      wa = p.W + ((int64_t)e * p.N + n) * K;
      wb = p.W2 + ((int64_t)e * p.N + n) * K;
    } else {
      wa = p.W + ((int64_t)e * 2 * p.N + (n >> 4) * 32 + (n & 15)) * K;
      wb = wa + (int64_t)16 * K;
    }
  } else {
    wa = p.W + ((int64_t)e * p.N + min(n0 + li, p.N - 1)) * K;
    wb = p.W + ((int64_t)e * p.N + min(n0 + 16 + li, p.N - 1)) * K;
  }
  wa += 8 * g, wb += 8 * g;
  const int nk = K >> 5, per = ((nk + 7) >> 3) * 2, s1 = min(nk, (w + 1) * per);  // (a wave starts at a line)
  f32x4 aa = {0.f, 0.f, 0.f, 0.f}, ab = aa;
  for (int s = w * per; s < s1; s += U) {
    s16x8 fx[U], fa[U], fb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + u, s1 - 1) * 32;
      fa[u] = *reinterpret_cast<const s16x8*>(wa + k);
      fb[u] = *reinterpret_cast<const s16x8*>(wb + k);
      fx[u] = *reinterpret_cast<const s16x8*>(x + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s1) {
        aa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[u], fx[u], aa, 0, 0, 0);
        ab = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[u], fx[u], ab, 0, 0, 0);
      }
  }
  *reinterpret_cast<f32x4*>(&part[w][0][li][4 * g]) = aa;
  *reinterpret_cast<f32x4*>(&part[w][1][li][4 * g]) = ab;
  __syncthreads();
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
  if (r >= rows) return;
  float va = 0.f, vb = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    va += part[i][0][r][c];
    vb += part[i][1][r][c];
  }
  const float sw = MODE != MD_DOWN && p.pw ? p.pw[p.order[row0 + r]] : 1.f;
  const int64_t at = (int64_t)(row0 + r) * p.N + n0 + c;
  if constexpr (MODE == MD_GLU) {
    if (n0 + c < p.N) ((bf16_t*)p.C)[at] = f2bf(glu_clamped_t(va * sw, vb * sw, p.limit, p.alpha, p.silu));
  } else if constexpr (MODE == MD_GELU) {
    if (n0 + c < p.N) ((bf16_t*)p.C)[at] = f2bf(gelu_erf(va * sw));
    if (n0 + 16 + c < p.N) ((bf16_t*)p.C)[at + 16] = f2bf(gelu_erf(vb * sw));
  } else {
    if (n0 + c < p.N) ((float*)p.C)[at] = va;
    if (n0 + 16 + c < p.N) ((float*)p.C)[at + 16] = vb;
  }
}

// mode 0: act [pairs, N] = glu(X W^T, X W2^T) (W2 null: gate and up rows of W [E, 2 N, K] in alternating groups of 16), 1: gelu(X W^T),
// rows of X gathered through order / top; 2: C = X W^T in fp32, rows of X in expert order
void launch_moe_dec(int mode, const void* X, int64_t ldx, const void* W, const void* W2, const void* meta, const void* order, void* C,
                    int E, int maxt, int top, int N, int K, float limit, float alpha, const void* pw, int silu, hipStream_t st) {
  if (maxt <= 0) return;
  if (mode < 0 || mode > 2) throw std::runtime_error("moe_dec: mode");
  if (K % 32 || K <= 0 || N <= 0 || ldx % 8 || (((uintptr_t)X | (uintptr_t)W | (uintptr_t)W2) & 15))
    throw std::runtime_error("moe_dec: K % 32, rows of 16-byte alignment");
  if (mode == MD_GLU && !W2 && N % 16) throw std::runtime_error("moe_dec: gate and up in groups of 16 rows");
  if (maxt > 65535) throw std::runtime_error("moe_dec: too many row tiles");
  MoeDecArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, (const bf16_t*)W2, C, N, K, (const int*)meta, (const int*)order,
               (const float*)pw, E, maxt, top, silu, limit, alpha};
  const int bn = mode == MD_GLU ? 16 : 32;
  dim3 g((N + bn - 1) / bn, maxt);
  if (mode == MD_GLU) moe_dec_kernel<MD_GLU><<<g, 256, 0, st>>>(a);
  else if (mode == MD_GELU) moe_dec_kernel<MD_GELU><<<g, 256, 0, st>>>(a);
  else moe_dec_kernel<MD_DOWN><<<g, 256, 0, st>>>(a);
  HIP_CHECK_LAUNCH();
}
