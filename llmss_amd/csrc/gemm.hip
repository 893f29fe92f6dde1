// Tensor-parallel linear layers on MFMA (reference: F.linear -> cuBLAS
// in FastLinear/TensorParallel{Column,Row}Linear, utils/layers.py:39-179, with bias and
// activation as separate ATen kernels).
//
//   Y[M, N] = epilogue( X[M, K] . W[N, K]^T )    X, W bf16 (W optionally fp8-e4m3 + per-row scale)
//   epilogue: (* w_scale[n]) (+ bias[n]) then act (gelu_tanh | gelu | relu) or SwiGLU
//   SwiGLU ("silu_glu"): W rows are interleaved in 16-row groups at load time, group 2p = gate
//   rows [16p, 16p+16), group 2p+1 = up rows [16p, 16p+16); the kernel writes
//   Y[:, 16p + i] = silu(gate) * up (or the tanh form of GELU), so the [M, 2F] intermediate never reaches HBM.
//
// Kernel family (launch_gemm picks one per call; explicit hints and the autotuned plan table,
// ops/autotune.py, override the static planner):
//  * gemm_stream / gemm_stream2 (M <= 16, fp8 decode candidates): weight streaming straight into
//    VGPRs (non-temporal), X staged once per chunk in LDS, 3-deep register ring, split-K slabs.
//  * gemm_tiled<BM, BN, NS, WNT, F8> (decode / mid M): 64x64, 64x128 or 128x128 tiles, 4 waves,
//    both operands by global_load_lds into XOR-swizzled 128-B-row LDS images, an NS-stage ring
//    (2-6) waited with counted vmcnt across raw barriers, split-K over grid.y with fp32 slabs that
//    the NEXT kernel sums (add_norm, rope) or splitk_reduce; F8 = fp8 weight tiles (W8A16).
//  * gemm_streamk: persistent stream-K variant of the tiled kernel (in-kernel last-arriver combine).
//  * gemm_big<F8> (prefill, M >= ~1K): 256x256 tile, 8 waves, 128 KiB double buffer whose K-tile
//    t+2 is restaged while t is still being multiplied; F8 = W8A8 on the MX-fp8 matrix cores.
//  * gemm_f8f8: tiled W8A8 for fp8 shapes too small for the 256x256 tile.
// Split-K partial slabs never leave a call unless gemm_partial_slabs() says so (one source of
// truth shared with the Python wrapper).
#include "common.h"
#include "gemm_quad.h"

#include <mutex>
#include <unordered_map>

// -------------------------------------------------------------------------------------------
// helpers
// -------------------------------------------------------------------------------------------
// 16 fp8-e4m3 (one 16-B word) -> two bf16x8 fragments
__device__ __forceinline__ void fp8x16_to_bf16(const u32x4& w, s16x8& f0, s16x8& f1) {
  const unsigned wd[4] = {w[0], w[1], w[2], w[3]};
  short o[16];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(wd[q], false);
    f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(wd[q], true);
    o[4 * q + 0] = (short)f2bf(lo[0]);
    o[4 * q + 1] = (short)f2bf(lo[1]);
    o[4 * q + 2] = (short)f2bf(hi[0]);
    o[4 * q + 3] = (short)f2bf(hi[1]);
  }
  f0 = s16x8{o[0], o[1], o[2], o[3], o[4], o[5], o[6], o[7]};
  f1 = s16x8{o[8], o[9], o[10], o[11], o[12], o[13], o[14], o[15]};
}

__device__ __forceinline__ float epi_value(float v, int n, const float* wscale, const bf16_t* bias, int act) {
  if (wscale) v *= wscale[n];
  if (bias) v += bf2f(bias[n]);
  return apply_act(v, act);
}

// -------------------------------------------------------------------------------------------
// weight-streaming GEMM (M <= 128: decode / small batches)
// grid (ceil(N / (64*NT)), SPLITK), block 256 = 4 waves; wave w owns NT 16-column tiles.
// Per K-chunk of KC: X[0:16*MT, chunk] is staged ONCE per workgroup into LDS by 16-byte
// global_load_lds (lane-linear image, XOR swizzle applied on the source address: rule 21), and
// shared by the 4 waves; each wave streams its W rows straight into VGPRs (non-temporal: read
// once per step), 32 B per lane = a full 128-B line per 4 lanes. W for chunk c+1 and X for chunk
// c+1 are issued before the MFMAs of chunk c (register ring of 2 named buffers, static indexing).
// -------------------------------------------------------------------------------------------
template <int MT, int NT, int KC, bool FP8W>
struct StreamCfg {
  static constexpr int ROWS = MT * 16;
  static constexpr int RB = KC * 2;                     // LDS row bytes
  static constexpr int XBYTES = ROWS * RB;              // one X chunk
  static constexpr int NG = KC / 64;                    // 64-k groups per chunk
  static constexpr int WV = FP8W ? 1 : 2;               // u32x4 per lane per (nt, group)
  static constexpr int SW = (KC / 8 - 1) < 15 ? (KC / 8 - 1) : 15;  // swizzle mask (chunks)
  static constexpr int XINST = XBYTES / 1024 / 4;       // glds per wave per chunk
  static_assert(XBYTES % 4096 == 0, "X chunk must be a multiple of 4 KiB (4 waves x 1 KiB)");
};

template <int MT, int NT, int KC, bool FP8W>
__device__ __forceinline__ void stream_stage_x(const bf16_t* __restrict__ X, int64_t ldx, int M, int K, int kc0,
                                               char* xbuf, int w, int lane) {
  using C = StreamCfg<MT, NT, KC, FP8W>;
#pragma unroll
  for (int i = 0; i < C::XINST; ++i) {
    const int inst = i * 4 + w;
    const int o = inst * 1024 + lane * 16;
    const int row = o / C::RB;
    const int pc = (o % C::RB) >> 4;
    const int gc = pc ^ (row & C::SW);
    const int k = min(kc0 + gc * 8, K - 8);
    const bf16_t* src = X + (int64_t)min(row, M - 1) * ldx + k;
    __builtin_amdgcn_global_load_lds((const void*)src, (LDS_AS void*)(xbuf + inst * 1024), 16, 0, 0);
  }
}

template <int MT, int NT, int KC, bool FP8W>
__device__ __forceinline__ void stream_load_w(const char* const (&wrow)[NT], int kc0, int K, int g,
                                              u32x4 (&wr)[NT][KC / 64][FP8W ? 1 : 2]) {
  constexpr int WB = FP8W ? 1 : 2;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int q = 0; q < KC / 64; ++q) {
      int k = kc0 + 64 * q + 16 * g;
      k = k < K ? k : 0;  // tail lanes read a valid address; their fragments are zeroed at use
      const u32x4* p = reinterpret_cast<const u32x4*>(wrow[nt] + (int64_t)k * WB);
      wr[nt][q][0] = __builtin_nontemporal_load(p);
      if constexpr (!FP8W) wr[nt][q][1] = __builtin_nontemporal_load(p + 1);
    }
}

// 8 fp8-e4m3 (two dwords) -> one bf16x8 fragment
__device__ __forceinline__ s16x8 fp8x8_to_bf16(unsigned w0, unsigned w1) {
  const f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8(w0, false), b = __builtin_amdgcn_cvt_pk_f32_fp8(w0, true);
  const f32x2 c = __builtin_amdgcn_cvt_pk_f32_fp8(w1, false), d = __builtin_amdgcn_cvt_pk_f32_fp8(w1, true);
  return s16x8{(short)f2bf(a[0]), (short)f2bf(a[1]), (short)f2bf(b[0]), (short)f2bf(b[1]),
               (short)f2bf(c[0]), (short)f2bf(c[1]), (short)f2bf(d[0]), (short)f2bf(d[1])};
}

template <int MT, int NT, int KC, bool FP8W, bool TAIL>
__device__ __forceinline__ void stream_compute(const char* xbuf, const u32x4 (&wr)[NT][KC / 64][FP8W ? 1 : 2],
                                               f32x4 (&acc)[MT][NT], int kc0, int K, int li, int g) {
  using C = StreamCfg<MT, NT, KC, FP8W>;
  const s16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < C::NG; ++q) {
    const bool ok = !TAIL || (kc0 + 64 * q + 16 * g < K);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      s16x8 b[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if constexpr (FP8W) b[nt] = fp8x8_to_bf16(wr[nt][q][0][2 * s], wr[nt][q][0][2 * s + 1]);
        else b[nt] = *reinterpret_cast<const s16x8*>(&wr[nt][q][s]);
        if (TAIL && !ok) b[nt] = z;
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int r = mt * 16 + li;
        const int c = 8 * q + 2 * g + s;
        s16x8 a = *reinterpret_cast<const s16x8*>(xbuf + r * C::RB + ((c ^ (r & C::SW)) << 4));
        if (TAIL && !ok) a = z;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[nt], acc[mt][nt], 0, 0, 0);
      }
    }
  }
}

template <int MT, int NT, int KC, bool FP8W>
__global__ __launch_bounds__(256, 2) void gemm_stream_kernel(const bf16_t* __restrict__ X, int64_t ldx,
                                                             const void* __restrict__ Wv, int64_t ldw,
                                                             const float* __restrict__ wscale,
                                                             const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                             int64_t ldy, float* __restrict__ part, int M, int N, int K,
                                                             int act, int glu) {
  using C = StreamCfg<MT, NT, KC, FP8W>;
  __shared__ __attribute__((aligned(16))) char xs[2 * C::XBYTES];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (64 * NT) + w * (16 * NT);
  const int split = blockIdx.y, nsplit = gridDim.y;
  const int nck = (K + KC - 1) / KC;
  const int cb = (int)((int64_t)nck * split / nsplit), ce = (int)((int64_t)nck * (split + 1) / nsplit);

  f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  constexpr int WB = FP8W ? 1 : 2;
  const char* wrow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    wrow[nt] = (const char*)Wv + (int64_t)min(n0 + nt * 16 + li, N - 1) * ldw * WB;  // + k*WB per load

  u32x4 wA[NT][KC / 64][FP8W ? 1 : 2], wB[NT][KC / 64][FP8W ? 1 : 2];
  const bool tail_k = (K % KC) != 0;
  if (cb < ce) {
    stream_stage_x<MT, NT, KC, FP8W>(X, ldx, M, K, cb * KC, xs, w, lane);
    stream_load_w<MT, NT, KC, FP8W>(wrow, cb * KC, K, g, wA);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  for (int c = cb; c < ce; c += 2) {
    // ---- even chunk: compute from wA / buffer 0, prefetch chunk c+1 into wB / buffer 1
    if (c + 1 < ce) {
      stream_stage_x<MT, NT, KC, FP8W>(X, ldx, M, K, (c + 1) * KC, xs + C::XBYTES, w, lane);
      stream_load_w<MT, NT, KC, FP8W>(wrow, (c + 1) * KC, K, g, wB);
    }
    if (tail_k && c == nck - 1) stream_compute<MT, NT, KC, FP8W, true>(xs, wA, acc, c * KC, K, li, g);
    else stream_compute<MT, NT, KC, FP8W, false>(xs, wA, acc, c * KC, K, li, g);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (c + 1 >= ce) break;
    // ---- odd chunk: compute from wB / buffer 1, prefetch chunk c+2 into wA / buffer 0
    if (c + 2 < ce) {
      stream_stage_x<MT, NT, KC, FP8W>(X, ldx, M, K, (c + 2) * KC, xs, w, lane);
      stream_load_w<MT, NT, KC, FP8W>(wrow, (c + 2) * KC, K, g, wA);
    }
    if (tail_k && c + 1 == nck - 1) stream_compute<MT, NT, KC, FP8W, true>(xs + C::XBYTES, wB, acc, (c + 1) * KC, K, li, g);
    else stream_compute<MT, NT, KC, FP8W, false>(xs + C::XBYTES, wB, acc, (c + 1) * KC, K, li, g);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  // ---- epilogue (C layout: col = lane&15 -> n, row = 4*(lane>>4)+i -> m) --------------------
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mt * 16 + 4 * g + i;
      if (m >= M) continue;
      if (nsplit > 1) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int n = n0 + nt * 16 + li;
          if (n < N) part[((int64_t)split * M + m) * N + n] = acc[mt][nt][i] * (wscale ? wscale[n] : 1.f);
        }
      } else if (glu) {
#pragma unroll
        for (int p = 0; p < NT / 2; ++p) {
          const int ng = n0 + 2 * p * 16 + li, nu = ng + 16;
          if (nu < N) {
            const float gv = epi_value(acc[mt][2 * p][i], ng, wscale, bias, ACT_NONE);
            const float uv = epi_value(acc[mt][2 * p + 1][i], nu, wscale, bias, ACT_NONE);
            Y[(int64_t)m * ldy + n0 / 2 + p * 16 + li] = f2bf(glu_gate(gv, act) * uv);
          }
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int n = n0 + nt * 16 + li;
          if (n < N) Y[(int64_t)m * ldy + n] = f2bf(epi_value(acc[mt][nt][i], n, wscale, bias, act));
        }
      }
    }
  }
}

// -------------------------------------------------------------------------------------------
// weight-streaming GEMM, v2: register-staged X + 3-deep W register ring (2 chunks in flight).
// v1 stages X with global_load_lds; while an LDS-DMA is in flight hipcc drains vmcnt(0) at every
// use of an ordinary load (guide §5 'Pipelining across barriers'), which caps v1 at ONE W chunk
// in flight per wave. Here every load is an ordinary global_load, issued in the order
// X(c+1), W(c+2) before the MFMAs of chunk c, so the compiler's counted vmcnt waits only for what
// each consumer needs: the ds_write of X(c+1) waits for X(c+1), not for W(c+2).
// Same tile/K mapping as v1 (verified by tests/test_kernel_emulation.py), same epilogue.
// -------------------------------------------------------------------------------------------
template <int MT, int NT, int KC, bool FP8W>
struct Stream2Cfg {
  static constexpr int ROWS = MT * 16;
  static constexpr int RB = KC * 2;
  static constexpr int XBYTES = ROWS * RB;
  static constexpr int CPR = KC / 8;                      // 16-B chunks per X row
  static constexpr int XPT = ROWS * CPR / 256;            // X chunks per thread per K-chunk
  static constexpr int SW = (CPR - 1) < 15 ? (CPR - 1) : 15;
  static_assert((ROWS * CPR) % 256 == 0, "X chunk must split evenly over 256 threads");
};

template <int MT, int NT, int KC, bool FP8W>
__device__ __forceinline__ void stream2_load_x(const bf16_t* __restrict__ X, int64_t ldx, int M, int K, int kc0,
                                               u32x4 (&xr)[Stream2Cfg<MT, NT, KC, FP8W>::XPT]) {
  using C = Stream2Cfg<MT, NT, KC, FP8W>;
#pragma unroll
  for (int i = 0; i < C::XPT; ++i) {
    const int id = threadIdx.x + i * 256;
    const int row = id / C::CPR, c = id % C::CPR;
    const int k = min(kc0 + c * 8, K - 8);
    xr[i] = *reinterpret_cast<const u32x4*>(X + (int64_t)min(row, M - 1) * ldx + k);
  }
}

template <int MT, int NT, int KC, bool FP8W>
__device__ __forceinline__ void stream2_store_x(char* xbuf, const u32x4 (&xr)[Stream2Cfg<MT, NT, KC, FP8W>::XPT]) {
  using C = Stream2Cfg<MT, NT, KC, FP8W>;
#pragma unroll
  for (int i = 0; i < C::XPT; ++i) {
    const int id = threadIdx.x + i * 256;
    const int row = id / C::CPR, c = id % C::CPR;
    *reinterpret_cast<u32x4*>(xbuf + row * C::RB + ((c ^ (row & C::SW)) << 4)) = xr[i];
  }
}

template <int MT, int NT, int KC, bool FP8W>
__global__ __launch_bounds__(256, 2) void gemm_stream2_kernel(const bf16_t* __restrict__ X, int64_t ldx,
                                                              const void* __restrict__ Wv, int64_t ldw,
                                                              const float* __restrict__ wscale,
                                                              const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                              int64_t ldy, float* __restrict__ part, int M, int N,
                                                              int K, int act, int glu) {
  using C = Stream2Cfg<MT, NT, KC, FP8W>;
  __shared__ __attribute__((aligned(16))) char xs[2 * C::XBYTES];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (64 * NT) + w * (16 * NT);
  const int split = blockIdx.y, nsplit = gridDim.y;
  const int nck = (K + KC - 1) / KC;
  const int cb = (int)((int64_t)nck * split / nsplit), ce = (int)((int64_t)nck * (split + 1) / nsplit);

  f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int WB = FP8W ? 1 : 2;
  const char* wrow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) wrow[nt] = (const char*)Wv + (int64_t)min(n0 + nt * 16 + li, N - 1) * ldw * WB;

  u32x4 w0[NT][KC / 64][FP8W ? 1 : 2], w1[NT][KC / 64][FP8W ? 1 : 2], w2[NT][KC / 64][FP8W ? 1 : 2];
  u32x4 xr[C::XPT];
  const bool tail_k = (K % KC) != 0;
  if (cb < ce) {
    stream2_load_x<MT, NT, KC, FP8W>(X, ldx, M, K, cb * KC, xr);
    stream_load_w<MT, NT, KC, FP8W>(wrow, cb * KC, K, g, w0);
    if (cb + 1 < ce) stream_load_w<MT, NT, KC, FP8W>(wrow, (cb + 1) * KC, K, g, w1);
    stream2_store_x<MT, NT, KC, FP8W>(xs, xr);
    __syncthreads();
  }
  // Steady state: branch-free steps (every prefetch valid), so hipcc's vmcnt bookkeeping stays
  // exact and it waits only for the chunk being consumed (a load under an `if` makes the counts
  // path-dependent and the compiler then drains vmcnt(0) before re-issuing - measured).
#define STREAM2_STEADY(CUR, NXT2)                                                                             \
  {                                                                                                          \
    stream2_load_x<MT, NT, KC, FP8W>(X, ldx, M, K, (c + 1) * KC, xr);                                        \
    stream_load_w<MT, NT, KC, FP8W>(wrow, (c + 2) * KC, K, g, NXT2);                                         \
    __builtin_amdgcn_sched_barrier(0); /* keep the prefetch ahead of the MFMAs (hipcc sinks it) */           \
    stream_compute<MT, NT, KC, FP8W, false>(xs + ((c - cb) & 1) * C::XBYTES, CUR, acc, c * KC, K, li, g);    \
    __builtin_amdgcn_sched_barrier(0);                                                                       \
    stream2_store_x<MT, NT, KC, FP8W>(xs + ((c + 1 - cb) & 1) * C::XBYTES, xr);                              \
    __syncthreads();                                                                                         \
    ++c;                                                                                                     \
  }
#define STREAM2_REM(CUR, NXT2)                                                                                \
  {                                                                                                          \
    if (c >= ce) break;                                                                                      \
    if (c + 1 < ce) stream2_load_x<MT, NT, KC, FP8W>(X, ldx, M, K, (c + 1) * KC, xr);                        \
    if (c + 2 < ce) stream_load_w<MT, NT, KC, FP8W>(wrow, (c + 2) * KC, K, g, NXT2);                         \
    const char* xb = xs + ((c - cb) & 1) * C::XBYTES;                                                        \
    if (tail_k && c == nck - 1) stream_compute<MT, NT, KC, FP8W, true>(xb, CUR, acc, c * KC, K, li, g);      \
    else stream_compute<MT, NT, KC, FP8W, false>(xb, CUR, acc, c * KC, K, li, g);                            \
    if (c + 1 < ce) stream2_store_x<MT, NT, KC, FP8W>(xs + ((c + 1 - cb) & 1) * C::XBYTES, xr);              \
    __syncthreads();                                                                                         \
    ++c;                                                                                                     \
  }
  int c = cb;
  for (; c + 4 < ce;) {  // 3 chunks per iteration; chunks c+2..c+4 exist -> all prefetches valid
    STREAM2_STEADY(w0, w2)
    STREAM2_STEADY(w1, w0)
    STREAM2_STEADY(w2, w1)
  }
  do {  // remaining <= 4 chunks (ring rotation continues at w0); also handles the K tail chunk
    STREAM2_REM(w0, w2)
    STREAM2_REM(w1, w0)
    STREAM2_REM(w2, w1)
    STREAM2_REM(w0, w2)
  } while (0);
#undef STREAM2_STEADY
#undef STREAM2_REM

#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mt * 16 + 4 * g + i;
      if (m >= M) continue;
      if (nsplit > 1) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int n = n0 + nt * 16 + li;
          if (n < N) part[((int64_t)split * M + m) * N + n] = acc[mt][nt][i] * (wscale ? wscale[n] : 1.f);
        }
      } else if (glu) {
#pragma unroll
        for (int p = 0; p < NT / 2; ++p) {
          const int ng = n0 + 2 * p * 16 + li, nu = ng + 16;
          if (nu < N) {
            const float gv = epi_value(acc[mt][2 * p][i], ng, wscale, bias, ACT_NONE);
            const float uv = epi_value(acc[mt][2 * p + 1][i], nu, wscale, bias, ACT_NONE);
            Y[(int64_t)m * ldy + n0 / 2 + p * 16 + li] = f2bf(glu_gate(gv, act) * uv);
          }
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int n = n0 + nt * 16 + li;
          if (n < N) Y[(int64_t)m * ldy + n] = f2bf(epi_value(acc[mt][nt][i], n, wscale, bias, act));
        }
      }
    }
  }
}

// split-K reduction + epilogue: part [S, M, N] fp32 (w_scale already applied). The slabs are read in groups of 8 with
// every load of a group issued before its adds (one memory round trip per group, not per slab; adds in slab order).
__device__ __forceinline__ float slab_sum(const float* __restrict__ part, int S, int64_t stride, int64_t off) {
  constexpr int SG = 8;
  float v = 0.f;
  for (int s0 = 0; s0 < S; s0 += SG) {
    float x[SG];
#pragma unroll
    for (int g = 0; g < SG; ++g) x[g] = part[(int64_t)min(s0 + g, S - 1) * stride + off];
#pragma unroll
    for (int g = 0; g < SG; ++g) v += s0 + g < S ? x[g] : 0.f;
  }
  return v;
}

__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S, int M, int N,
                                                            const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                            int64_t ldy, int act, int glu) {
  const int m = blockIdx.y;
  const int nout = glu ? N / 2 : N;
  const int64_t stride = (int64_t)M * N;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nout; c += gridDim.x * blockDim.x) {
    if (glu) {
      const int p = c >> 4, i = c & 15;
      const int ng = 32 * p + i, nu = ng + 16;
      float gv = slab_sum(part, S, stride, (int64_t)m * N + ng), uv = slab_sum(part, S, stride, (int64_t)m * N + nu);
      if (bias) { gv += bf2f(bias[ng]); uv += bf2f(bias[nu]); }
      Y[(int64_t)m * ldy + c] = f2bf(glu_gate(gv, act) * uv);
    } else {
      float v = slab_sum(part, S, stride, (int64_t)m * N + c);
      if (bias) v += bf2f(bias[c]);
      Y[(int64_t)m * ldy + c] = f2bf(apply_act(v, act));
    }
  }
}

// -------------------------------------------------------------------------------------------
// tiled GEMM (prefill / large M), bf16 weights. Tile BM x BN x 64, 4 waves in 2x2, each wave
// (BM/2) x (BN/2) = MTW x NTW mfma_f32_16x16x32 accumulators. Both operands staged by 16-byte
// global_load_lds into an XOR-swizzled image (chunk ^= row & 7: conflict-free ds_read_b128),
// double-buffered; XCD-aware tile order (T1). The tile is chosen per call so small-N tensor-
// parallel shards still produce >= ~256 workgroups (128x128, 64x128 or 64x64).
// -------------------------------------------------------------------------------------------
constexpr int TBK = 64;

// F8: B (weights) is fp8-e4m3, one byte per element: its LDS image is [BN][64 B] with the 16-B chunk
// q of row r stored at q ^ ((r >> 2) & 3) (ds_read_b64 fragment reads conflict-free, bank-simulated).
template <int BN, bool F8, int NW = 4>
struct TiledB {
  static constexpr int ROWB = F8 ? 64 : 128;  // LDS bytes per B row per 64-k stage
  static constexpr int BYTES = BN * ROWB;
  static constexpr int LOADS = F8 ? BN / (16 * NW) : BN / (8 * NW);  // glds per wave per stage
};

template <int BM, int BN, bool WNT = false, bool F8 = false, int NW = 4>
__device__ __forceinline__ void tiled_stage(const bf16_t* __restrict__ A, int64_t lda, int M, const void* __restrict__ Bv,
                                            int64_t ldb, int N, int K, int m0, int n0, int k0, char* sA, char* sB,
                                            int w, int lane) {
  // one wave-instruction = 1 KiB = 8 rows x 128 B; A needs BM/8 of them, B BN/8 (NW waves share)
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile rows must split evenly over the waves");
#pragma unroll
  for (int it = 0; it < BM / (8 * NW); ++it) {
    const int inst = it * NW + w;
    const int row = inst * 8 + (lane >> 3);
    const int c = (lane & 7) ^ (row & 7);
    const int kc = min(k0 + c * 8, K - 8);
    const bf16_t* ga = A + (int64_t)min(m0 + row, M - 1) * lda + kc;
    __builtin_amdgcn_global_load_lds((const void*)ga, (LDS_AS void*)(sA + inst * 1024), 16, 0, 0);
  }
  if constexpr (F8) {
    const unsigned char* B = reinterpret_cast<const unsigned char*>(Bv);
#pragma unroll
    for (int it = 0; it < BN / (16 * NW); ++it) {  // one wave-instruction = 16 rows x 64 B
      const int inst = it * NW + w;
      const int row = inst * 16 + (lane >> 2);
      const int gq = (lane & 3) ^ ((row >> 2) & 3);
      const int kc = min(k0 + gq * 16, K - 16);
      const unsigned char* gb = B + (int64_t)min(n0 + row, N - 1) * ldb + kc;
      __builtin_amdgcn_global_load_lds((const void*)gb, (LDS_AS void*)(sB + inst * 1024), 16, 0, WNT ? 2 : 0);
    }
  } else {
    const bf16_t* B = reinterpret_cast<const bf16_t*>(Bv);
#pragma unroll
    for (int it = 0; it < BN / (8 * NW); ++it) {
      const int inst = it * NW + w;
      const int row = inst * 8 + (lane >> 3);
      const int c = (lane & 7) ^ (row & 7);
      const int kc = min(k0 + c * 8, K - 8);
      const bf16_t* gb = B + (int64_t)min(n0 + row, N - 1) * ldb + kc;
      // weights read once per step (single M tile): non-temporal (aux = 2), guide 'nt-weights'
      __builtin_amdgcn_global_load_lds((const void*)gb, (LDS_AS void*)(sB + inst * 1024), 16, 0, WNT ? 2 : 0);
    }
  }
}

template <int MTW, int NTW, bool MASK, bool F8 = false>
__device__ __forceinline__ void tiled_compute(const char* sA, const char* sB, f32x4 (&acc)[MTW][NTW], int wr, int wc,
                                              int li, int g, int k0, int K) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int c = 4 * s + g;
    const bool valid = !MASK || (k0 + c * 8 < K);
    const s16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    s16x8 a[MTW], b[NTW];
#pragma unroll
    for (int t = 0; t < MTW; ++t) {
      const int ra = wr * (MTW * 16) + t * 16 + li;
      a[t] = *reinterpret_cast<const s16x8*>(sA + ra * 128 + ((c ^ (ra & 7)) << 4));
      if (MASK && !valid) a[t] = z;
    }
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      const int rb = wc * (NTW * 16) + t * 16 + li;
      if constexpr (F8) {  // k bytes [32 s + 8 g, +8) = half (g & 1) of 16-B chunk 2 s + g / 2
        const int pq = (2 * s + (g >> 1)) ^ ((rb >> 2) & 3);
        const u32x2 raw = *reinterpret_cast<const u32x2*>(sB + rb * 64 + pq * 16 + (g & 1) * 8);
        b[t] = fp8x8_to_bf16(raw[0], raw[1]);
      } else {
        b[t] = *reinterpret_cast<const s16x8*>(sB + rb * 128 + ((c ^ (rb & 7)) << 4));
      }
      if (MASK && !valid) b[t] = z;
    }
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], b[nt], acc[mt][nt], 0, 0, 0);
  }
}

// s_waitcnt vmcnt(N) with expcnt / lgkmcnt left alone (gfx9 encoding: vmcnt[3:0] + [15:14])
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// wait until at most min(younger, MAXY) stages of LOADS instructions each are outstanding
template <int LOADS, int MAXY>
__device__ __forceinline__ void wait_vmcnt_upto(int younger) {
  if constexpr (MAXY <= 0) {
    wait_vmcnt<0>();
  } else {
    if (younger >= MAXY) wait_vmcnt<LOADS * MAXY>();
    else wait_vmcnt_upto<LOADS, MAXY - 1>(younger);
  }
}

// Barrier that lets global_load_lds stay in flight across it: __syncthreads()' release fence
// would emit vmcnt(0) and drain the prefetch (guide: "Pipelining across barriers").
__device__ __forceinline__ void lds_barrier() {
  // lgkmcnt(0) through the builtin (vmcnt / expcnt at their maxima), which the compiler's wait-count
  // pass accounts for: after an inline-asm wait it still believes earlier LDS reads are pending and
  // adds an lgkmcnt(0) in front of the next MFMA that uses their registers
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// NW = 4: waves 2 (M) x 2 (N); NW = 8 (256-row tiles, one workgroup per CU): waves 4 (M) x 2 (N),
// each 64 x BN/2 - mid-M shapes (TP-sharded decode at M = 256-512) are per-CU load-latency bound,
// so a wider tile moves fewer bytes per output through each CU's load path (guide: "Projection GEMM
// at M = 256").
template <int BM, int BN, int NS, bool WNT, bool F8 = false, int NW = 4>
__global__ __launch_bounds__(64 * NW) void gemm_tiled_kernel(const bf16_t* __restrict__ A, int64_t lda,
                                                         const void* __restrict__ B, int64_t ldb,
                                                         const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                         int64_t ldy, float* __restrict__ part, int M, int N, int K,
                                                         int act, int glu, const float* __restrict__ wscale,
                                                         int* __restrict__ cnt, QkvEpi qe) {
  constexpr int MTW = BM / (8 * NW), NTW = BN / 32;  // 16x16 tiles per wave (waves NW/2 x 2)
  constexpr int A_BYTES = BM * TBK * 2, B_BYTES = TiledB<BN, F8, NW>::BYTES, STAGE = A_BYTES + B_BYTES;
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wr = w >> 1, wc = w & 1;
  const int ntn = (N + BN - 1) / BN, ntm = (M + BM - 1) / BM;
  const TileWork tw = tile_work(ntm, ntn, BM, BN);
  const int m0 = tw.m0, n0 = tw.n0, zk = tw.z;

  f32x4 acc[MTW][NTW];
#pragma unroll
  for (int a = 0; a < MTW; ++a)
#pragma unroll
    for (int b = 0; b < NTW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // split-K (grid.y): slice z covers k-tiles [t0, t1); partial sums go to part[z] (fp32)
  const int nk_all = (K + TBK - 1) / TBK;
  const int per = (nk_all + gridDim.y - 1) / gridDim.y;
  const int t0 = zk * per, t1 = min(nk_all, t0 + per);
  if constexpr (NS == 2) {
    if (t0 < t1) {
      tiled_stage<BM, BN, WNT, F8, NW>(A, lda, M, B, ldb, N, K, m0, n0, t0 * TBK, smem, smem + A_BYTES, w, lane);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    for (int t = t0; t < t1; ++t) {
      const int cur = (t - t0) & 1;
      char* nA = smem + (cur ^ 1) * STAGE;
      char* cA = smem + cur * STAGE;
      if (t + 1 < t1) tiled_stage<BM, BN, WNT, F8, NW>(A, lda, M, B, ldb, N, K, m0, n0, (t + 1) * TBK, nA, nA + A_BYTES, w, lane);
      if (t + 1 == nk_all && (K % TBK)) tiled_compute<MTW, NTW, true, F8>(cA, cA + A_BYTES, acc, wr, wc, li, g, t * TBK, K);
      else tiled_compute<MTW, NTW, false, F8>(cA, cA + A_BYTES, acc, wr, wc, li, g, t * TBK, K);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  } else {
    // NS-stage ring: stage t+NS-1 is issued while stage t is computed; the wait before compute
    // only covers stage t (the younger stages' LOADS instructions each stay in flight): no drain.
    constexpr int LOADS = BM / (8 * NW) + TiledB<BN, F8, NW>::LOADS;  // global_load_lds per wave per stage
#pragma unroll
    for (int j = 0; j < NS - 1; ++j)
      if (t0 + j < t1)
        tiled_stage<BM, BN, WNT, F8, NW>(A, lda, M, B, ldb, N, K, m0, n0, (t0 + j) * TBK, smem + j * STAGE,
                            smem + j * STAGE + A_BYTES, w, lane);
    int cur = 0;
    for (int t = t0; t < t1; ++t) {
      wait_vmcnt_upto<LOADS, NS - 2>(t1 - 1 - t);  // stages younger than t still in flight
      lds_barrier();  // stage t visible; every wave is past compute(t-1), so its buffer is free
      char* cA = smem + cur * STAGE;
      const int nxt = cur == 0 ? NS - 1 : cur - 1;  // (cur + NS - 1) % NS
      if (t + NS - 1 < t1) {
        char* nA = smem + nxt * STAGE;
        tiled_stage<BM, BN, WNT, F8, NW>(A, lda, M, B, ldb, N, K, m0, n0, (t + NS - 1) * TBK, nA, nA + A_BYTES, w, lane);
      }
      if (t + 1 == nk_all && (K % TBK)) tiled_compute<MTW, NTW, true, F8>(cA, cA + A_BYTES, acc, wr, wc, li, g, t * TBK, K);
      else tiled_compute<MTW, NTW, false, F8>(cA, cA + A_BYTES, acc, wr, wc, li, g, t * TBK, K);
      cur = cur == NS - 1 ? 0 : cur + 1;
    }
  }
  // cnt: split-K slices combine in this launch (common.h splitk_combine); the last arriver of the
  // tile finishes it with the normal bf16 epilogue, the others are done
  if (cnt) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!splitk_combine<MTW, NTW>(acc, part, cnt, (n0 / BN) * ntm + m0 / BM, gridDim.y, zk, w, NW, lane,
                                  reinterpret_cast<int*>(smem)))
      return;
    part = nullptr;
  }
  if constexpr (!F8) {
    // QKV projection (RoPE + paged KV write) runs in the LDS-staged epilogue
    // (unsplit / combined plans only)
    if (qe.D) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      tile_store_lds<BM, BN, MTW, NTW, 64 * NW, NS * STAGE>(acc, smem, wr * (MTW * 16), wc * (NTW * 16), m0, n0, M,
                                                             N, nullptr, Y, ldy, bias, act, glu, qe);
      return;
    }
  }
  // epilogue (C layout: col = lane&15 -> n, row = 4*(lane>>4)+i -> m)
  const int wn0 = n0 + wc * (NTW * 16);
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + wr * (MTW * 16) + mt * 16 + 4 * g + i;
      if (m >= M) continue;
      if (part) {
        float* pr = part + ((int64_t)zk * M + m) * N;
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          const int n = wn0 + nt * 16 + li;
          if (n < N) pr[n] = F8 ? acc[mt][nt][i] * wscale[n] : acc[mt][nt][i];
        }
      } else if (glu) {
#pragma unroll
        for (int p = 0; p < NTW / 2; ++p) {
          const int ng = wn0 + 2 * p * 16 + li, nu = ng + 16;
          if (nu < N) {
            float gv = acc[mt][2 * p][i], uv = acc[mt][2 * p + 1][i];
            if constexpr (F8) { gv *= wscale[ng]; uv *= wscale[nu]; }
            if (bias) { gv += bf2f(bias[ng]); uv += bf2f(bias[nu]); }
            Y[(int64_t)m * ldy + wn0 / 2 + p * 16 + li] = f2bf(glu_gate(gv, act) * uv);
          }
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          const int n = wn0 + nt * 16 + li;
          if (n < N) {
            float v = acc[mt][nt][i];
            if constexpr (F8) v *= wscale[n];
            if (bias) v += bf2f(bias[n]);
            Y[(int64_t)m * ldy + n] = f2bf(apply_act(v, act));
          }
        }
      }
    }
  }
}

// -------------------------------------------------------------------------------------------
// W8A8 big-tile GEMM (fp8 prefill, M >= ~1024; bf16 prompt batches take gemm_quad.hip or gemm_pp_kernel below):
// 256x256 tile of 128-element fp8 K-tiles, 8 waves (2 x 4), each wave 128x64 = 8x4 accumulators on the
// MX-fp8 16x16x128 MFMA. LDS = 2 buffers x {A rows 0-127, A rows 128-255, B rows 0-127, B rows 128-255}
// of 16 KiB = 128 KiB -> one workgroup per CU.
// Per K-tile t: (1) counted vmcnt(8) retires stage t while stage t+1 stays in flight, raw
// barrier; (2) every wave reads ALL its fragments of tile t into VGPRs (24 ds_read_b128) and
// runs the first half of its MFMAs; (3) barrier (lgkmcnt(0): all reads of buffer t&1 done) and
// stage t+2 is issued into that same buffer, then the second half of MFMAs. Prefetch distance
// is therefore ~1.5 K-tiles of MFMA time and no barrier ever drains the DMA queue (guide:
// "Pipelining across barriers", 3-buffer-equivalent depth in 2 buffers).
// Requires K % 64 == 0; rows beyond M / N are clamped on load and masked on store.
// -------------------------------------------------------------------------------------------
// M-tiles per tile group of the big-tile kernel's launch order (gemm_big_set_group; measured 4)
static int g_big_group_m = 4;
void gemm_big_set_group(int g) { g_big_group_m = g >= 1 && g <= 64 ? g : 4; }

// one MX-fp8 16x16x128 MFMA from two 16-B fragment halves per operand (unit E8M0 block scales)
__device__ __forceinline__ f32x4 mfma_f8x2(s16x8 a0, s16x8 a1, s16x8 b0, s16x8 b1, f32x4 c) {
  typedef int __attribute__((ext_vector_type(4))) i32x4_t;
  typedef int __attribute__((ext_vector_type(8))) i32x8_t;
  const i32x4_t al = __builtin_bit_cast(i32x4_t, a0), ah = __builtin_bit_cast(i32x4_t, a1);
  const i32x4_t bl = __builtin_bit_cast(i32x4_t, b0), bh = __builtin_bit_cast(i32x4_t, b1);
  const i32x8_t av = __builtin_shufflevector(al, ah, 0, 1, 2, 3, 4, 5, 6, 7);
  const i32x8_t bv = __builtin_shufflevector(bl, bh, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 0, 0, 0, 127, 0, 127);
}

// F8: both operands fp8-e4m3 (W8A8): a 128-element fp8 K-tile has exactly the byte layout of the
// 64-element bf16 one, so staging / LDS image / fragment addresses are shared; each (m, n) takes one
// MX-fp8 16x16x128 MFMA per K-tile (the two 16-B chunks 2g, 2g+1 of the lane's row), and the
// per-token x per-channel scales are applied in the epilogue.
template <bool F8>
__global__ __launch_bounds__(512, 1) void gemm_big_kernel(const void* __restrict__ A, int64_t lda,
                                                          const void* __restrict__ B, int64_t ldb,
                                                          const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                          int64_t ldy, int M, int N, int K, int act, int glu,
                                                          const float* __restrict__ xs, const float* __restrict__ ws,
                                                          int group_m) {
  constexpr int ES = F8 ? 1 : 2;  // operand bytes per element
  constexpr int HALF = 16384, BUF = 4 * HALF;
  __shared__ __attribute__((aligned(16))) char smem[2 * BUF];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wr = w >> 2, wc = w & 3;
  const int ntn = (N + 255) / 256, ntm = (M + 255) / 256;
  // XCD-contiguous tile ranges, grouped GM M-tiles high: the 32 workgroups an XCD runs at once cover a
  // 4 x 8 block of tiles, so its L2 fills 4 A + 8 B panels per round instead of ~1 A + 32 B panels
  // (PMC: 4 TB/s of L2 fills and 47 % of wave cycles waiting before this)
  const int GM = group_m;
  const int tile = xcd_remap(blockIdx.x, ntn * ntm);
  const int grp = tile / (GM * ntn), gidx = tile - grp * (GM * ntn);
  const int gm = min(GM, ntm - grp * GM);
  const int m0 = (grp * GM + gidx % gm) * 256, n0 = (gidx / gm) * 256;
  const int nk = K * ES / 128;  // 128-byte K-tiles

  // staging: half h (0,1: A rows 128h.., 2,3: B rows 128(h-2)..), 2 x 1-KiB glds per wave; lane ->
  // row inst*8 + lane/8, LDS chunk lane&7 holding global chunk (lane&7) ^ (row&7) (swizzle on source)
  const char* src[4] = {(const char*)A, (const char*)A, (const char*)B, (const char*)B};
  const int64_t ld[4] = {lda * ES, lda * ES, ldb * ES, ldb * ES};  // bytes
  int64_t soff[4][2];
  int lofs[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int inst = i * 8 + w;
    const int row = inst * 8 + (lane >> 3);
    const int gc = (lane & 7) ^ (row & 7);
    lofs[i] = inst * 1024;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const bool isA = h < 2;
      const int lim = isA ? M : N;
      const int r = min((isA ? m0 : n0) + (h & 1) * 128 + row, lim - 1);
      soff[h][i] = (int64_t)r * ld[h] + gc * 16;
    }
  }
  auto stage = [&](int t, char* buf) {
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        __builtin_amdgcn_global_load_lds((const void*)(src[h] + soff[h][i] + (int64_t)t * 128),
                                         (LDS_AS void*)(buf + h * HALF + lofs[i]), 16, 0, 0);
  };

  f32x4 acc[8][4];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // fragment read offsets (bytes within a buffer): A half wr, B half wc>>1 (+64 rows for odd wc)
  int aoff[8][2], boff[4][2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    // bf16: k-half s; fp8: the lane's two 16-B chunks g, g + 4 (the same k permutation for A and B, the
    // conflict-free bf16 read pattern; chunks 2g, 2g + 1 hit the same banks)
    const int c = 4 * s + g;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int r = m * 16 + li;
      aoff[m][s] = wr * HALF + r * 128 + ((c ^ (r & 7)) << 4);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int r = (wc & 1) * 64 + n * 16 + li;
      boff[n][s] = (2 + (wc >> 1)) * HALF + r * 128 + ((c ^ (r & 7)) << 4);
    }
  }

  stage(0, smem);
  if (nk > 1) stage(1, smem + BUF);
  for (int t = 0; t < nk; ++t) {
    char* cur = smem + (t & 1) * BUF;
    if (t + 1 < nk) wait_vmcnt<8>();
    else wait_vmcnt<0>();
    lds_barrier();  // stage t landed for every wave
    s16x8 a[8][2], b[4][2];
    {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int n = 0; n < 4; ++n) b[n][s] = *reinterpret_cast<const s16x8*>(cur + boff[n][s]);
#pragma unroll
      for (int m = 0; m < 8; ++m) a[m][s] = *reinterpret_cast<const s16x8*>(cur + aoff[m][s]);
    }
    __builtin_amdgcn_s_setprio(1);
    if constexpr (F8) {  // first half: n-tiles 0, 1
#pragma unroll
      for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[m][n] = mfma_f8x2(a[m][0], a[m][1], b[n][0], b[n][1], acc[m][n]);
    } else {
#pragma unroll
      for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m][0], b[n][0], acc[m][n], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    }
    lds_barrier();  // every wave's reads of this buffer are complete -> restage it
    if (t + 2 < nk) stage(t + 2, cur);
    __builtin_amdgcn_s_setprio(1);
    if constexpr (F8) {  // second half: n-tiles 2, 3
#pragma unroll
      for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int n = 2; n < 4; ++n) acc[m][n] = mfma_f8x2(a[m][0], a[m][1], b[n][0], b[n][1], acc[m][n]);
    } else {
#pragma unroll
      for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m][1], b[n][1], acc[m][n], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // epilogue (C layout: col = lane&15 -> n, row = 4*(lane>>4)+i -> m)
  const int wn0 = n0 + wc * 64;
#pragma unroll
  for (int m = 0; m < 8; ++m) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = m0 + wr * 128 + m * 16 + 4 * g + i;
      if (row >= M) continue;
      const float sx = F8 ? xs[row] : 1.f;
      if (glu) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int ng = wn0 + 2 * p * 16 + li, nu = ng + 16;
          if (nu < N) {
            float gv = acc[m][2 * p][i], uv = acc[m][2 * p + 1][i];
            if constexpr (F8) { gv *= sx * ws[ng]; uv *= sx * ws[nu]; }
            if (bias) { gv += bf2f(bias[ng]); uv += bf2f(bias[nu]); }
            Y[(int64_t)row * ldy + wn0 / 2 + p * 16 + li] = f2bf(glu_gate(gv, act) * uv);
          }
        }
      } else {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const int col = wn0 + n * 16 + li;
          if (col < N) {
            float v = acc[m][n][i];
            if constexpr (F8) v *= sx * ws[col];
            if (bias) v += bf2f(bias[col]);
            Y[(int64_t)row * ldy + col] = f2bf(apply_act(v, act));
          }
        }
      }
    }
  }
}

// -------------------------------------------------------------------------------------------
// Ping-pong prefill GEMM (bf16, M >= ~1024) for what gemm_quad.hip does not take: K off 64 (Llama-2-7B's TP=8 down projection,
// K = 1376), N off 8 (GLU 32), rows over more than 31 bits of bytes (256 of them; gathered ones: all).
// 256x256x64 tile, 8 waves = two groups of 4 (waves 0-3 / 4-7; one wave of each group per SIMD). Waves
// 4-7 pass one extra barrier before the K-loop, so on every SIMD one wave's compute segment runs beside
// its partner's load segment (guide "The 256^2 8-phase template", MI355X_MICROARCH "Two waves per SIMD").
//   * LDS = 2 buffers x 4 slots of 16 KiB: slot 0 = A half 0, 1 = B half 0, 2 = B half 1, 3 = A half 1.
//     A half h holds block rows {128 r + 64 h + i}, B half h block columns {64 c + 32 h + j}, so each
//     wave's contiguous 128x64 output splits into four 64x32 quadrants Q(mq, nq) reading A slot mq and
//     B slot nq. Rows are 128 B (one K-tile), chunk-XOR swizzled on the source address (rule 21).
//   * 4 phases per K-tile: Q(0,0) [reads A0 + B0: 12 ds_read_b128], Q(0,1) [B1: 4], Q(1,1) [A1: 8],
//     Q(1,0) [B0 still in registers]. Phase = load segment (2 LDS-DMA of slot p of the NEXT K-tile, then
//     the fragment reads, then a counted vmcnt) | barrier | 16 MFMA 16x16x32 | barrier.
//   * RAW: a slot is read one phase after the vmcnt that retires it (vmcnt 4/4/6/4 in steady state,
//     2/0 on the last K-tile); WAR: a slot is restaged >= 4 phases after its last read.
//   * waves 4-7 run at s_setprio 1 (the arbitration loser of each pair, MI355X_MICROARCH item 4).
// Measured vs the previous 2-barrier kernel at M = 8192 (Llama-2-7B shapes, random data, one process):
// +4-13 %; the no-stagger control equals the old kernel. Ablations (profiles/r5_gemm_pp/README.md): the
// LDS-DMA + fragment-read traffic through the LDS costs ~25 % each on top of the MFMA/barrier skeleton.
// K % 8 == 0: a partial last K-tile reads zeros (zpage) for the chunks past K; rows beyond M / N are clamped on load
// and masked on store.
// GRP: the grouped expert products of a mixture-of-experts layer (moe.hip's tile list, tiles of 256 rows): 1 - rows of A
// gathered through order[] / top, activation in the epilogue, bf16 rows in expert order; 2 - A rows already in expert
// order, fp32 output. Every die takes a contiguous run of the list's tiles with all their column tiles.
// -------------------------------------------------------------------------------------------
__device__ __forceinline__ void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int GRP>
__global__ __launch_bounds__(512, 1) void gemm_pp_kernel(const bf16_t* __restrict__ A, int64_t lda,
                                                         const bf16_t* __restrict__ B, int64_t ldb,
                                                         const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                         int64_t ldy, int M, int N, int K, int act, int glu,
                                                         int group_m, const char* __restrict__ zpage, PpGroup gr) {
  constexpr int SLOT = 16384, BUF = 4 * SLOT;
  __shared__ __attribute__((aligned(16))) char smem[2 * BUF];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wr = w >> 2, wc = w & 3;
  const int ntn = (N + 255) / 256, ntm = (M + 255) / 256;
  const int GM = group_m;  // XCD-contiguous tile ranges, GM M-tiles per group (as gemm_big)
  int m0, n0;
  if constexpr (GRP != 0) {
    const int nt = gr.meta[0];
    if ((int)blockIdx.x >= nt * ntn) return;
    const int id = xcd_remap(blockIdx.x, nt * ntn), ty = id / ntn;
    const int e = gr.meta[1 + (gr.E + 1) + ty];
    n0 = (id - ty * ntn) * 256;
    m0 = gr.meta[1 + (gr.E + 1) + gr.maxt + ty];
    M = gr.meta[1 + e + 1];
    B += (int64_t)e * gr.sB;
  } else {
    const int tile = xcd_remap(blockIdx.x, ntn * ntm);
    const int grp = tile / (GM * ntn), gidx = tile - grp * (GM * ntn);
    const int gm = min(GM, ntm - grp * GM);
    m0 = (grp * GM + gidx % gm) * 256, n0 = (gidx / gm) * 256;
  }
  const int nk = (K + 63) / 64;

  // staging: slot h, instruction i (0, 1) = 8 local rows x 128 B, local row lr = (8 i + w) * 8 + lane / 8;
  // LDS chunk lane & 7 holds global chunk (lane & 7) ^ (lr & 7)
  const char* src[4] = {(const char*)A, (const char*)B, (const char*)B, (const char*)A};
  int64_t soff[4][2];
  int lofs[2], kcol[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int inst = i * 8 + w;
    const int lr = inst * 8 + (lane >> 3);
    const int gc = (lane & 7) ^ (lr & 7);
    lofs[i] = inst * 1024;
    kcol[i] = gc * 8;
    int ar0 = min(m0 + (lr >> 6) * 128 + (lr & 63), M - 1);
    int ar1 = min(m0 + (lr >> 6) * 128 + 64 + (lr & 63), M - 1);
    if constexpr (GRP == 1) ar0 = gr.order[ar0] / gr.top, ar1 = gr.order[ar1] / gr.top;
    const int bc0 = min(n0 + (lr >> 5) * 64 + (lr & 31), N - 1);
    const int bc1 = min(n0 + (lr >> 5) * 64 + 32 + (lr & 31), N - 1);
    soff[0][i] = (int64_t)ar0 * lda * 2 + gc * 16;
    soff[3][i] = (int64_t)ar1 * lda * 2 + gc * 16;
    soff[1][i] = (int64_t)bc0 * ldb * 2 + gc * 16;
    soff[2][i] = (int64_t)bc1 * ldb * 2 + gc * 16;
  }
  auto stage = [&](int t, int h, char* buf) {
    const bool last = t == nk - 1;  // wave-uniform
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const char* p = src[h] + soff[h][i] + (int64_t)t * 128;
      if (last) p = t * 64 + kcol[i] >= K ? zpage : p;  // chunks past K (of A and B) land as zeros
      __builtin_amdgcn_global_load_lds((const void*)p, (LDS_AS void*)(buf + h * SLOT + lofs[i]), 16, 0, 0);
    }
  };
  // fragment offsets inside a slot: A rows wr*64 + mt*16 + li, B rows wc*32 + nt*16 + li; k-half s -> chunk 4s+g
  // (the conflict-free ds_read_b128 image of gemm_big)
  int aoff[4][2], boff[2][2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int c = 4 * s + g;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int r = wr * 64 + mt * 16 + li;
      aoff[mt][s] = r * 128 + ((c ^ (r & 7)) << 4);
    }
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int r = wc * 32 + nt * 16 + li;
      boff[nt][s] = r * 128 + ((c ^ (r & 7)) << 4);
    }
  }
  f32x4 acc[8][4];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  s16x8 fa[4][2], fb0[2][2], fb1[2][2];
  auto rdA = [&](const char* slot) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int s = 0; s < 2; ++s) fa[mt][s] = *reinterpret_cast<const s16x8*>(slot + aoff[mt][s]);
  };
  auto rdB = [&](const char* slot, s16x8 (&fb)[2][2]) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int s = 0; s < 2; ++s) fb[nt][s] = *reinterpret_cast<const s16x8*>(slot + boff[nt][s]);
  };
  auto quad = [&](int mq, int nq, const s16x8 (&fb)[2][2]) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mq * 4 + mt][nq * 2 + nt] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[mt][s], fb[nt][s], acc[mq * 4 + mt][nq * 2 + nt], 0, 0, 0);
  };
  // one phase: LDS-DMA of slot h of the next K-tile, fragment reads, vmcnt(n) retiring what the next phase
  // reads, barrier, the quadrant's 16 MFMAs, barrier
  auto phase = [&](auto rd, int t, int h, bool more, int n_more, int n_last, int mq, int nq,
                   const s16x8 (&fb)[2][2]) {
    if (more) stage(t + 1, h, smem + ((t + 1) & 1) * BUF);
    rd();
    switch (more ? n_more : n_last) {
      case 0: wait_vmcnt<0>(); break;
      case 2: wait_vmcnt<2>(); break;
      case 4: wait_vmcnt<4>(); break;
      case 6: wait_vmcnt<6>(); break;
      default: break;
    }
    pp_barrier();
    quad(mq, nq, fb);
    pp_barrier();
  };

#pragma unroll
  for (int h = 0; h < 4; ++h) stage(0, h, smem);
  wait_vmcnt<4>();  // slots 0, 1 (A0, B0) of K-tile 0
  pp_barrier();
  if (w >= 4) {
    __builtin_amdgcn_s_setprio(1);
    pp_barrier();  // the stagger: waves 4-7 run one barrier behind waves 0-3
  }
  for (int t = 0; t < nk; ++t) {
    const char* cur = smem + (t & 1) * BUF;
    const bool more = t + 1 < nk;
    phase([&] { rdA(cur); rdB(cur + SLOT, fb0); }, t, 0, more, 4, 2, 0, 0, fb0);
    phase([&] { rdB(cur + 2 * SLOT, fb1); }, t, 1, more, 4, 0, 0, 1, fb1);
    phase([&] { rdA(cur + 3 * SLOT); }, t, 2, more, 6, -1, 1, 1, fb1);
    phase([&] {}, t, 3, more, 4, -1, 1, 0, fb0);
  }
  if (w < 4) pp_barrier();  // balances the stagger barrier
  __builtin_amdgcn_s_setprio(0);
  wait_vmcnt<0>();
  if constexpr (GRP == 2) {
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + wr * 128 + a * 16 + 4 * g + i;
        if (row >= M) continue;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int col = n0 + wc * 64 + b * 16 + li;
          if (col < N) gr.Yf[(int64_t)row * ldy + col] = acc[a][b][i];
        }
      }
  } else {
    tile_store_lds<256, 256, 8, 4, 512, 2 * BUF>(acc, smem, wr * 128, wc * 64, m0, n0, M, N, nullptr, Y, ldy, bias,
                                                 act, glu);
  }
}

// -------------------------------------------------------------------------------------------
// stream-K tiled GEMM (mid-size M: TP-sharded decode at M = 128-512, mid prefill). Split-K grids
// leave CUs unevenly loaded (e.g. 352 blocks on 256 CUs: some CUs run two, the rest one) and pay
// a reduce launch. Here a persistent grid of G workgroups splits the flattened (tile, k-step)
// iteration space into G equal contiguous ranges; the LDS ring of the tiled kernel runs straight
// across tile boundaries. A tile whose k-range spans several workgroups is combined in-kernel:
// every segment stores its fp32 accumulators (register layout, 16 B per lane, coalesced), then
// draws a ticket (agent-scope release fence + relaxed atomic, guide 'splitk-seam' recipe); the
// last arriver acquires, adds the other segments and runs the epilogue. Counters reset themselves.
// -------------------------------------------------------------------------------------------
__device__ __forceinline__ int sk_block_of(int64_t x, int64_t U, int G) {  // block whose range holds unit x
  int g = (int)((x * G) / U);
  while (g + 1 < G && (int64_t)(g + 1) * U / G <= x) ++g;
  while (g > 0 && (int64_t)g * U / G > x) --g;
  return g;
}

template <int MTW, int NTW>
__device__ __forceinline__ void tile_epilogue(const f32x4 (&acc)[MTW][NTW], bf16_t* __restrict__ Y, int64_t ldy,
                                              const bf16_t* __restrict__ bias, int M, int N, int m0, int n0, int wr,
                                              int wc, int li, int g, int act, int glu) {
  const int wn0 = n0 + wc * (NTW * 16);
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + wr * (MTW * 16) + mt * 16 + 4 * g + i;
      if (m >= M) continue;
      if (glu) {
#pragma unroll
        for (int p = 0; p < NTW / 2; ++p) {
          const int ng = wn0 + 2 * p * 16 + li, nu = ng + 16;
          if (nu < N) {
            float gv = acc[mt][2 * p][i], uv = acc[mt][2 * p + 1][i];
            if (bias) { gv += bf2f(bias[ng]); uv += bf2f(bias[nu]); }
            Y[(int64_t)m * ldy + wn0 / 2 + p * 16 + li] = f2bf(glu_gate(gv, act) * uv);
          }
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          const int n = wn0 + nt * 16 + li;
          if (n < N) {
            float v = acc[mt][nt][i];
            if (bias) v += bf2f(bias[n]);
            Y[(int64_t)m * ldy + n] = f2bf(apply_act(v, act));
          }
        }
      }
    }
  }
}

template <int BM, int BN, int NS, bool WNT>
__global__ __launch_bounds__(256) void gemm_streamk_kernel(const bf16_t* __restrict__ A, int64_t lda,
                                                           const bf16_t* __restrict__ B, int64_t ldb,
                                                           const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                           int64_t ldy, float* __restrict__ part,
                                                           int* __restrict__ counters, int maxseg, int M, int N, int K,
                                                           int act, int glu) {
  constexpr int MTW = BM / 32, NTW = BN / 32;
  constexpr int A_BYTES = BM * TBK * 2, B_BYTES = BN * TBK * 2, STAGE = A_BYTES + B_BYTES;
  constexpr int LOADS = BM / 32 + BN / 32;
  constexpr int TILE_F = BM * BN;  // fp32 per partial tile
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE + 16];  // + ticket broadcast (one LDS object)
  int* s_ticket = reinterpret_cast<int*>(smem + NS * STAGE);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wr = w >> 1, wc = w & 1;
  const int ntn = (N + BN - 1) / BN, ntm = (M + BM - 1) / BM;
  const int tiles = ntn * ntm, nk = (K + TBK - 1) / TBK;
  const int U = tiles * nk;  // host guarantees < 2^31
  const int G = gridDim.x;
  const int u0 = (int)((int64_t)blockIdx.x * U / G), u1 = (int)((int64_t)(blockIdx.x + 1) * U / G);
  if (u0 >= u1) return;

  // (tile, k-step) of the next unit to stage, advanced incrementally: no divisions in the k-loop
  int pf_t = u0 / nk, pf_k = u0 - (u0 / nk) * nk;
  int pf_m0 = (pf_t / ntn) * BM, pf_n0 = (pf_t % ntn) * BN;
  auto stage_next = [&](char* buf) {
    tiled_stage<BM, BN, WNT>(A, lda, M, B, ldb, N, K, pf_m0, pf_n0, pf_k * TBK, buf, buf + A_BYTES, w, lane);
    if (++pf_k == nk) {
      pf_k = 0;
      ++pf_t;
      pf_m0 = (pf_t / ntn) * BM;
      pf_n0 = (pf_t % ntn) * BN;
    }
  };

  f32x4 acc[MTW][NTW];
#pragma unroll
  for (int a = 0; a < MTW; ++a)
#pragma unroll
    for (int b = 0; b < NTW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int j = 0; j < NS - 1; ++j)
    if (u0 + j < u1) stage_next(smem + j * STAGE);
  int cur = 0;
  int t = u0 / nk, kk = u0 - (u0 / nk) * nk;  // unit being computed
  for (int u = u0; u < u1; ++u) {
    wait_vmcnt_upto<LOADS, NS - 2>(min(u1 - 1 - u, NS));
    lds_barrier();
    char* cA = smem + cur * STAGE;
    if (u + NS - 1 < u1) stage_next(smem + (cur == 0 ? NS - 1 : cur - 1) * STAGE);
    if (kk == nk - 1 && (K % TBK)) tiled_compute<MTW, NTW, true>(cA, cA + A_BYTES, acc, wr, wc, li, g, kk * TBK, K);
    else tiled_compute<MTW, NTW, false>(cA, cA + A_BYTES, acc, wr, wc, li, g, kk * TBK, K);
    cur = cur == NS - 1 ? 0 : cur + 1;

    if (u + 1 != u1 && kk != nk - 1) {  // segment continues
      ++kk;
      continue;
    }
    // ---- segment end: tile t, this workgroup's k-steps up to kk
    const int m0 = (t / ntn) * BM, n0 = (t % ntn) * BN;
    const int tu0 = t * nk;
    const bool whole = u0 <= tu0 && kk == nk - 1;
    if (whole) {
      tile_epilogue<MTW, NTW>(acc, Y, ldy, bias, M, N, m0, n0, wr, wc, li, g, act, glu);
    } else {
      const int gfirst = sk_block_of(tu0, U, G), glast = sk_block_of((int64_t)tu0 + nk - 1, U, G);
      const int nseg = glast - gfirst + 1, seg = (int)blockIdx.x - gfirst;
      float* pt = part + (int64_t)t * maxseg * TILE_F;
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt)
          *reinterpret_cast<f32x4*>(pt + (int64_t)seg * TILE_F + (((w * MTW + mt) * NTW + nt) * 64 + lane) * 4) =
              acc[mt][nt];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        *s_ticket = __hip_atomic_fetch_add(&counters[t], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (*s_ticket == nseg - 1) {  // last arriver: combine and finish the tile
        if (threadIdx.x == 0) {
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          counters[t] = 0;  // ready for the next launch
        }
        __syncthreads();
        for (int s2 = 0; s2 < nseg; ++s2) {
          if (s2 == seg) continue;
#pragma unroll
          for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) {
              const f32x4 o = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(
                  pt + (int64_t)s2 * TILE_F + (((w * MTW + mt) * NTW + nt) * 64 + lane) * 4));
#pragma unroll
              for (int i = 0; i < 4; ++i) acc[mt][nt][i] += o[i];
            }
        }
        tile_epilogue<MTW, NTW>(acc, Y, ldy, bias, M, N, m0, n0, wr, wc, li, g, act, glu);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stores / reads above must not count as ring stages
#pragma unroll
    for (int a = 0; a < MTW; ++a)
#pragma unroll
      for (int b = 0; b < NTW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    ++t;
    kk = 0;
  }
}

// -------------------------------------------------------------------------------------------
// W8A8 GEMM on the MX-fp8 matrix cores (Llama-2-70B in fp8, TP=8).
// Y = (Xq . Wq^T) * xs[m] * ws[n] (+ bias, act / SwiGLU): Xq = per-token fp8-e4m3 activations
// (quant_fp8_rows on X), Wq = per-channel fp8-e4m3 weights. The 16x16x128 f8f6f4 MFMA with unit
// block scales (E8M0 127) runs at the fp8 peak (2x bf16; the unscaled 16x16x32 fp8 form runs at
// the bf16 rate). Tiles: BM x BN x 128 bytes staged by glds into the same XOR-swizzled 128-B-row
// LDS image as the bf16 tiles; lane (r = l&15, g = l>>4) takes 32 bytes = k [32g, 32g+32) of its
// row as 2 x ds_read_b128. Used where fp8 GEMMs are compute-bound (prefill, M > 128).
// -------------------------------------------------------------------------------------------
typedef int __attribute__((ext_vector_type(8))) i32x8;
constexpr int TBK8 = 128;  // k (bytes) per stage

template <int BM, int BN>
__device__ __forceinline__ void f8_stage(const unsigned char* __restrict__ A, int64_t lda, int M,
                                         const unsigned char* __restrict__ B, int64_t ldb, int N, int K, int m0, int n0,
                                         int k0, char* sA, char* sB, int w, int lane) {
#pragma unroll
  for (int it = 0; it < BM / 32; ++it) {
    const int inst = it * 4 + w;
    const int row = inst * 8 + (lane >> 3);
    const int c = (lane & 7) ^ (row & 7);
    const int kc = min(k0 + c * 16, K - 16);
    __builtin_amdgcn_global_load_lds((const void*)(A + (int64_t)min(m0 + row, M - 1) * lda + kc),
                                     (LDS_AS void*)(sA + inst * 1024), 16, 0, 0);
  }
#pragma unroll
  for (int it = 0; it < BN / 32; ++it) {
    const int inst = it * 4 + w;
    const int row = inst * 8 + (lane >> 3);
    const int c = (lane & 7) ^ (row & 7);
    const int kc = min(k0 + c * 16, K - 16);
    __builtin_amdgcn_global_load_lds((const void*)(B + (int64_t)min(n0 + row, N - 1) * ldb + kc),
                                     (LDS_AS void*)(sB + inst * 1024), 16, 0, 0);
  }
}

template <int MTW, int NTW, bool MASK>
__device__ __forceinline__ void f8_compute(const char* sA, const char* sB, f32x4 (&acc)[MTW][NTW], int wr, int wc,
                                           int li, int g, int k0, int K) {
  // the lane's k-bytes: chunks g and g + 4 of the 128-byte step (one k permutation for A and B; the chunk
  // pattern of the bf16 reads, free of bank conflicts on the swizzled image)
  const bool v0 = !MASK || (k0 + 16 * g < K), v1 = !MASK || (k0 + 64 + 16 * g < K);
  i32x8 a[MTW], b[NTW];
#pragma unroll
  for (int t = 0; t < MTW; ++t) {
    const int r = wr * (MTW * 16) + t * 16 + li;
    const u32x4 lo = *reinterpret_cast<const u32x4*>(sA + r * 128 + ((g ^ (r & 7)) << 4));
    const u32x4 hi = *reinterpret_cast<const u32x4*>(sA + r * 128 + (((g + 4) ^ (r & 7)) << 4));
    a[t] = i32x8{(int)(v0 ? lo[0] : 0u), (int)(v0 ? lo[1] : 0u), (int)(v0 ? lo[2] : 0u), (int)(v0 ? lo[3] : 0u),
                 (int)(v1 ? hi[0] : 0u), (int)(v1 ? hi[1] : 0u), (int)(v1 ? hi[2] : 0u), (int)(v1 ? hi[3] : 0u)};
  }
#pragma unroll
  for (int t = 0; t < NTW; ++t) {
    const int r = wc * (NTW * 16) + t * 16 + li;
    const u32x4 lo = *reinterpret_cast<const u32x4*>(sB + r * 128 + ((g ^ (r & 7)) << 4));
    const u32x4 hi = *reinterpret_cast<const u32x4*>(sB + r * 128 + (((g + 4) ^ (r & 7)) << 4));
    b[t] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
  }
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt)
      acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[mt], b[nt], acc[mt][nt], 0, 0, 0, 127, 0, 127);
}

template <int BM, int BN, int NS>
__global__ __launch_bounds__(256) void gemm_f8f8_kernel(const unsigned char* __restrict__ A, int64_t lda,
                                                        const float* __restrict__ xs,
                                                        const unsigned char* __restrict__ B, int64_t ldb,
                                                        const float* __restrict__ ws,
                                                        const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                        int64_t ldy, float* __restrict__ part, int M, int N, int K,
                                                        int act, int glu) {
  constexpr int MTW = BM / 32, NTW = BN / 32;
  constexpr int A_BYTES = BM * TBK8, B_BYTES = BN * TBK8, STAGE = A_BYTES + B_BYTES;
  constexpr int LOADS = BM / 32 + BN / 32;
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wr = w >> 1, wc = w & 1;
  const int ntn = (N + BN - 1) / BN, ntm = (M + BM - 1) / BM;
  const TileWork tw = tile_work(ntm, ntn, BM, BN);
  const int m0 = tw.m0, n0 = tw.n0, zk = tw.z;
  f32x4 acc[MTW][NTW];
#pragma unroll
  for (int a = 0; a < MTW; ++a)
#pragma unroll
    for (int b = 0; b < NTW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nk_all = (K + TBK8 - 1) / TBK8;
  const int per = (nk_all + gridDim.y - 1) / gridDim.y;
  const int t0 = zk * per, t1 = min(nk_all, t0 + per);
#pragma unroll
  for (int j = 0; j < NS - 1; ++j)
    if (t0 + j < t1)
      f8_stage<BM, BN>(A, lda, M, B, ldb, N, K, m0, n0, (t0 + j) * TBK8, smem + j * STAGE, smem + j * STAGE + A_BYTES,
                       w, lane);
  int cur = 0;
  for (int t = t0; t < t1; ++t) {
    wait_vmcnt_upto<LOADS, NS - 2>(t1 - 1 - t);
    lds_barrier();
    char* cA = smem + cur * STAGE;
    if (t + NS - 1 < t1) {
      char* nA = smem + (cur == 0 ? NS - 1 : cur - 1) * STAGE;
      f8_stage<BM, BN>(A, lda, M, B, ldb, N, K, m0, n0, (t + NS - 1) * TBK8, nA, nA + A_BYTES, w, lane);
    }
    if (t + 1 == nk_all && (K % TBK8)) f8_compute<MTW, NTW, true>(cA, cA + A_BYTES, acc, wr, wc, li, g, t * TBK8, K);
    else f8_compute<MTW, NTW, false>(cA, cA + A_BYTES, acc, wr, wc, li, g, t * TBK8, K);
    cur = cur == NS - 1 ? 0 : cur + 1;
  }
  // epilogue: per-token x per-channel scales, then the usual bias / act / SwiGLU (or split-K slabs)
  const int wn0 = n0 + wc * (NTW * 16);
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + wr * (MTW * 16) + mt * 16 + 4 * g + i;
      if (m >= M) continue;
      const float sx = xs[m];
      if (part) {
        float* pr = part + ((int64_t)zk * M + m) * N;
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          const int n = wn0 + nt * 16 + li;
          if (n < N) pr[n] = acc[mt][nt][i] * sx * ws[n];
        }
      } else if (glu) {
#pragma unroll
        for (int p = 0; p < NTW / 2; ++p) {
          const int ng = wn0 + 2 * p * 16 + li, nu = ng + 16;
          if (nu < N) {
            float gv = acc[mt][2 * p][i] * sx * ws[ng], uv = acc[mt][2 * p + 1][i] * sx * ws[nu];
            if (bias) { gv += bf2f(bias[ng]); uv += bf2f(bias[nu]); }
            Y[(int64_t)m * ldy + wn0 / 2 + p * 16 + li] = f2bf(glu_gate(gv, act) * uv);
          }
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          const int n = wn0 + nt * 16 + li;
          if (n < N) {
            float v = acc[mt][nt][i] * sx * ws[n];
            if (bias) v += bf2f(bias[n]);
            Y[(int64_t)m * ldy + n] = f2bf(apply_act(v, act));
          }
        }
      }
    }
  }
}

// decode GEMM (csrc/gemm_dec.hip): hint tile bit 1024 (nt_hint bit 18), tile bits = the BN code, depth bits = ring
// depth code (2 / 3 / 4 / 4 stages per wave), split_hint = K split over the grid (fp32 slabs for the consumer)
void launch_gemm_dec(int code, int depth, const bf16_t* X, int64_t ldx, const void* W, int64_t ldw, const float* wscale,
                     const bf16_t* bias, bf16_t* Y, int64_t ldy, float* part, int M, int N, int K, int act, int glu,
                     int split, hipStream_t st, const QkvEpi* qe, int* cnt);
bool gemm_dec_bn(int code, int* bn);
bool gemm_dec_f8_ok(int code, int M);
// the decode GEMM's in-launch combine (hint bit 256 with a split) fits the workspace: [tile][split][64 * bn] fp32
static bool dec_combine_fits(int N, int tsel, int s, int64_t ws_bytes) {
  int bn;
  if (!(tsel & 256) || s <= 1 || !gemm_dec_bn(tsel & 15, &bn)) return false;
  return (int64_t)((N + bn - 1) / bn) * s * 64 * bn * 4 <= ws_bytes;
}
static constexpr int kDecHint = 1024;
static int dec_split(int M, int N, int K, int split_hint, int64_t ws_bytes) {
  int s = std::max(1, std::min(split_hint, (K + 63) / 64));
  if ((int64_t)s * M * N * 4 > ws_bytes) s = 1;
  return s;
}
static constexpr int kFourHint = 2048;
bool gemm_four_dims(int code, int* bm, int* bn);
bool gemm_four_ok(int N, int K, int64_t ldx, int64_t ldw, const void* Y, int64_t ldy, bool glu);
void launch_gemm_four(int code, const bf16_t* X, int64_t ldx, const bf16_t* W, int64_t ldw, const bf16_t* bias, bf16_t* Y, int64_t ldy, float* part,
                      int M, int N, int K, int act, int glu, int split, int group_m, hipStream_t st, int* cnt, const QkvEpi* qe);
bool gemm_mid_dims(int tsel, int* bm, int* bn, int* threads);
void launch_gemm_mid(int tsel, int depth, bool wnt, const bf16_t* X, int64_t ldx, const bf16_t* W, int64_t ldw,
                     const bf16_t* bias, bf16_t* Y, int64_t ldy, float* part, int M, int N, int K, int act, int glu,
                     int split, hipStream_t st, int* cnt = nullptr,
                     const QkvEpi* qe = nullptr, const float* xs = nullptr, const float* wsc = nullptr,
                     bool ilv = false, const unsigned char* asc = nullptr);

// tile: 1 = 128x128, 2 = 64x128, 3 = 64x64; ring depth 2-4; split-K over grid.y; 8-13: the gemm_mid tiles
// (buffer-descriptor staging, csrc/gemm_mid.hip, fp8 MFMA variant; K % 128 == 0; ilv: its software-pipelined
// k-loop, >= 3 stages)
// MX-fp8 activations (gemm_mid tiles only): asc = e8m0 scales [M][K / 32] of xq (xs unused: nullptr), and mxq / mxs =
// a SwiGLU output written as MX-fp8 instead of bf16 y (e4m3 [M][N / 2] with row stride ldy, scales [M][N / 64]; the
// output tile must hold whole 32-output blocks, BN % 64 == 0, and finish in the launch: no split)
// partial_out: a split plan without activation / GLU leaves its fp32 slabs [split, M, N] (scales applied, no
// bias) in `workspace` for the consumer (rope_cache / add_norm sum them) and returns the split; else 0.
int launch_gemm_f8f8(const void* xq, int64_t ldx, const void* xs, const void* wq, int64_t ldw, const void* wsc,
                     const void* bias, void* y, int64_t ldy, int M, int N, int K, int act, bool glu, int tile,
                     int depth, int split, void* workspace, int64_t ws_bytes, hipStream_t st, bool partial_out,
                     bool ilv, void* mxq, void* mxs, const void* asc) {
  if (M == 0 || N == 0) return 0;
  if (K % 16) throw std::runtime_error("gemm_f8f8: K must be a multiple of 16");
  if (glu && (N % 32)) throw std::runtime_error("gemm_f8f8: glu needs N % 32 == 0");
  if (!y && !partial_out && !mxq) throw std::runtime_error("gemm_f8f8: output required");
  int bm = tile == 1 ? 128 : 64, bn = tile == 3 ? 64 : 128, thr = 256;
  const bool mid = tile >= 7 && tile <= 15;
  if (mid) {
    if (K % 128) throw std::runtime_error("gemm_f8f8: gemm_mid tiles need K % 128 == 0");
    gemm_mid_dims(tile, &bm, &bn, &thr);
  }
  if ((asc || mxq) && !mid) throw std::runtime_error("gemm_f8f8: MX-fp8 activations need a gemm_mid tile (7-15)");
  if (asc && (xs || K % 128)) throw std::runtime_error("gemm_f8f8: MX scales replace xs; K % 128 == 0");
  if (mxq && (!mxs || !glu || act == ACT_GELU_TANH || bn % 64 || N % 128 || ldy != N / 2 || partial_out))
    throw std::runtime_error("gemm_f8f8: MX output needs SwiGLU, BN % 64 == 0, N % 128 == 0, dense rows, no slabs");
  const int tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  const int nk = (K + TBK8 - 1) / TBK8;
  if (tile == 4 || (tile == 0 && K % 128 == 0 && ((M + 255) / 256) * ((N + 255) / 256) >= 192)) {
    if (K % 128) throw std::runtime_error("gemm_f8f8: the 256x256 tile needs K % 128 == 0");
    gemm_big_kernel<true><<<((M + 255) / 256) * ((N + 255) / 256), 512, 0, st>>>(
        xq, ldx, wq, ldw, (const bf16_t*)bias, (bf16_t*)y, ldy, M, N, K, act, glu ? 1 : 0, (const float*)xs,
        (const float*)wsc, g_big_group_m);
    HIP_CHECK_LAUNCH();
    return 0;
  }
  if (tile == 0) {  // auto: 128x128 when it fills the chip, else 64x128 / 64x64, split to >= ~256 WGs
    tile = ((M + 127) / 128) * ((N + 127) / 128) >= 240 ? 1 : (((M + 63) / 64) * ((N + 127) / 128) >= 240 ? 2 : 3);
    return launch_gemm_f8f8(xq, ldx, xs, wq, ldw, wsc, bias, y, ldy, M, N, K, act, glu, tile, depth, split, workspace,
                            ws_bytes, st, partial_out, ilv, mxq, mxs, asc);
  }
  if (split <= 0) {
    split = 1;
    while (tiles * split * 2 <= 512 && nk / (2 * split) >= 4 && split < 8) split *= 2;
  }
  split = std::max(1, std::min(split, nk));
  if ((int64_t)split * M * N * 4 > ws_bytes) split = 1;
  if (mxq && split > 1) throw std::runtime_error("gemm_f8f8: an MX-fp8 SwiGLU output cannot be split over K");
  float* part = split > 1 ? (float*)workspace : nullptr;
  const int act_k = split > 1 ? 0 : act, g = glu ? 1 : 0, glu_k = split > 1 ? 0 : g;
  if (depth <= 0) depth = tile == 1 ? 3 : 4;
  if (tile == 1 && depth > 3) depth = 3;
  dim3 grid(tiles, split);
  auto A = (const unsigned char*)xq;
  auto Bw = (const unsigned char*)wq;
  auto XS = (const float*)xs;
  auto WSc = (const float*)wsc;
  auto Bi = (const bf16_t*)bias;
  auto Y = (bf16_t*)y;
#define LF(BM_, BN_, NS_) \
  gemm_f8f8_kernel<BM_, BN_, NS_><<<grid, 256, 0, st>>>(A, ldx, XS, Bw, ldw, WSc, Bi, Y, ldy, part, M, N, K, act_k, glu_k)
  if (mid) {
    QkvEpi mx{};
    mx.mxq = (unsigned char*)mxq;
    mx.mxs = (unsigned char*)mxs;
    launch_gemm_mid(tile, depth, M <= bm, (const bf16_t*)xq, ldx, (const bf16_t*)wq, ldw, Bi, Y, ldy, part, M, N, K,
                    act_k, glu_k, split, st, nullptr, mxq ? &mx : nullptr, XS, WSc, ilv,
                    (const unsigned char*)asc);
  } else if (tile == 1) {
    if (depth >= 3) LF(128, 128, 3); else LF(128, 128, 2);
  } else if (tile == 2) {
    if (depth >= 4) LF(64, 128, 4); else if (depth == 3) LF(64, 128, 3); else LF(64, 128, 2);
  } else {
    if (depth >= 4) LF(64, 64, 4); else if (depth == 3) LF(64, 64, 3); else LF(64, 64, 2);
  }
#undef LF
  HIP_CHECK_LAUNCH();
  if (split > 1 && partial_out && !glu && act == 0) return split;
  if (split > 1) {
    if (!y) throw std::runtime_error("gemm_f8f8: output required");
    const int nout = glu ? N / 2 : N;
    dim3 rgrid(std::min((nout + 255) / 256, 64), M);
    splitk_reduce_kernel<<<rgrid, 256, 0, st>>>(part, split, M, N, Bi, Y, ldy, act, g);
    HIP_CHECK_LAUNCH();
  }
  return 0;
}

// the split a W8A8 call with these arguments leaves as slabs under partial_out (0 = finished output)
int gemm_f8f8_partial_slabs(int M, int N, int K, bool glu, int act, int tile, int split, int64_t ws_bytes) {
  if (M == 0 || N == 0 || glu || act != 0) return 0;
  if (tile == 4 || (tile == 0 && K % 128 == 0 && ((M + 255) / 256) * ((N + 255) / 256) >= 192)) return 0;
  if (tile == 0)
    tile = ((M + 127) / 128) * ((N + 127) / 128) >= 240 ? 1 : (((M + 63) / 64) * ((N + 127) / 128) >= 240 ? 2 : 3);
  int bm = tile == 1 ? 128 : 64, bn = tile == 3 ? 64 : 128, thr;
  if (tile >= 7 && tile <= 15) gemm_mid_dims(tile, &bm, &bn, &thr);
  const int tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  const int nk = (K + TBK8 - 1) / TBK8;
  if (split <= 0) {
    split = 1;
    while (tiles * split * 2 <= 512 && nk / (2 * split) >= 4 && split < 8) split *= 2;
  }
  split = std::max(1, std::min(split, nk));
  if ((int64_t)split * M * N * 4 > ws_bytes) split = 1;
  return split > 1 ? split : 0;
}

// -------------------------------------------------------------------------------------------
// host dispatch
// -------------------------------------------------------------------------------------------
template <int MT, int NT, int KC, bool FP8W, int VARIANT>
static void launch_stream_t(const bf16_t* X, int64_t ldx, const void* W, int64_t ldw, const float* ws, const bf16_t* bias,
                            bf16_t* Y, int64_t ldy, float* part, int M, int N, int K, int act, int glu, int splitk,
                            hipStream_t st) {
  dim3 grid((N + 64 * NT - 1) / (64 * NT), splitk);
  if constexpr (VARIANT == 2)
    gemm_stream2_kernel<MT, NT, KC, FP8W><<<grid, 256, 0, st>>>(X, ldx, W, ldw, ws, bias, Y, ldy, part, M, N, K, act, glu);
  else
    gemm_stream_kernel<MT, NT, KC, FP8W><<<grid, 256, 0, st>>>(X, ldx, W, ldw, ws, bias, Y, ldy, part, M, N, K, act, glu);
  HIP_CHECK_LAUNCH();
}

template <bool FP8W>
static void launch_stream(int variant, int mt, int nt, const bf16_t* X, int64_t ldx, const void* W, int64_t ldw,
                          const float* ws, const bf16_t* bias, bf16_t* Y, int64_t ldy, float* part, int M, int N, int K,
                          int act, int glu, int splitk, hipStream_t st) {
  if (variant == 2) {  // v2 instantiations (3-deep W ring): NT <= 2, spill-free at 2 waves/SIMD
#define LS2(MT_, NT_, KC_) \
  launch_stream_t<MT_, NT_, KC_, FP8W, 2>(X, ldx, W, ldw, ws, bias, Y, ldy, part, M, N, K, act, glu, splitk, st)
    if (nt >= 2) {
      if (mt == 1) LS2(1, 2, 128); else if (mt == 2) LS2(2, 2, 128); else if (mt <= 4) LS2(4, 2, 128); else LS2(8, 2, 64);
    } else {
      if (mt == 1) LS2(1, 1, 256); else if (mt == 2) LS2(2, 1, 128); else if (mt <= 4) LS2(4, 1, 128); else LS2(8, 1, 128);
    }
#undef LS2
    return;
  }
#define LS(MT_, NT_, KC_) \
  launch_stream_t<MT_, NT_, KC_, FP8W, 1>(X, ldx, W, ldw, ws, bias, Y, ldy, part, M, N, K, act, glu, splitk, st)
  // only register-feasible (spill-free at 2 waves/SIMD) instantiations
  if constexpr (FP8W) {
    if (nt >= 2) {
      if (mt == 1) LS(1, 2, 256); else if (mt == 2) LS(2, 2, 128); else if (mt <= 4) LS(4, 2, 128); else LS(8, 2, 64);
    } else {
      if (mt == 1) LS(1, 1, 256); else if (mt == 2) LS(2, 1, 256); else if (mt <= 4) LS(4, 1, 256); else LS(8, 1, 128);
    }
  } else {
    if (nt >= 4 && mt <= 2) {
      if (mt == 1) LS(1, 4, 128); else LS(2, 4, 128);
    } else if (nt >= 2) {
      if (mt == 1) LS(1, 2, 256); else if (mt == 2) LS(2, 2, 256); else if (mt <= 4) LS(4, 2, 256); else LS(8, 2, 64);
    } else {
      if (mt == 1) LS(1, 1, 256); else if (mt == 2) LS(2, 1, 256); else if (mt <= 4) LS(4, 1, 256); else LS(8, 1, 128);
    }
  }
#undef LS
}

// Tile/split choice for the streaming kernel: columns per workgroup and K splits such that the
// grid reaches ~2 workgroups per CU (256 CUs) without splitting K below 4 chunks per slice.
void gemm_stream_plan(int M, int N, int K, int* nt_out, int* splitk_out) {
  int nt = (N >= 16384) ? 2 : 1;
  const int nblk = (N + 64 * nt - 1) / (64 * nt);
  const int kc = M > 64 ? 128 : 256;
  const int nck = (K + kc - 1) / kc;
  // measured (bench/gemm_bench.py --sweep, Llama-2-7B shapes): M <= 16 likes ~3 workgroups per
  // CU, larger M ~1 per CU (its X tile already costs LDS); N alone filling the chip -> no split
  const int target = nblk >= 256 ? nblk : (M <= 16 ? 768 : 256);
  int s = 1;
  while (nblk * s < target && s < 16 && nck / (2 * s) >= 4) s *= 2;
  *nt_out = nt;
  *splitk_out = s;
}

int gemm_skinny_splitk(int M, int N, int K) {
  int nt, s;
  gemm_stream_plan(M, N, K, &nt, &s);
  return s;
}

int launch_tiled(const bf16_t* X, int64_t ldx, const void* W, int64_t ldw, const bf16_t* B, bf16_t* Y, int64_t ldy,
                 int M, int N, int K, int act, int g, int tsel, int split_hint, void* workspace, int64_t ws_bytes,
                 bool partial_out, hipStream_t st, const float* wscale = nullptr, const QkvEpi* qe = nullptr);

void gemm_tiled_plan(int M, int N, int K, int* tsel_io, int* split_io, bool glu);
void gemm_stream_plan(int M, int N, int K, int* nt_out, int* splitk_out);

// Returns the number of fp32 partial slabs [S, M, N] left in `workspace` (partial_out and the
// planner chose split-K: the consumer - add_norm - reduces them and adds `bias`), or 0 when Y
// holds the finished bf16 output.
// Autotuned plans: (M, N, K, glu, fp8) -> (nt_hint, split) measured by llmss_amd/ops/autotune.py
// for the shapes an engine will actually run (decode batch buckets x layer GEMMs). Consulted by
// every call without explicit hints and by gemm_plan, so split-K partial fusion stays consistent.
namespace {
std::mutex g_tuned_mu;
std::unordered_map<uint64_t, std::pair<int, int>> g_tuned;
// kind: 0 = bf16 [N, K] weights, 1 = fp8 weights, 3 = QKV
// RoPE / KV-write epilogue (launch_gemm_qkv)
uint64_t tune_key(int M, int N, int K, bool glu, int kind) {
  return ((uint64_t)(kind & 7) << 61) | ((uint64_t)(M & 0x7FFFF) << 42) | ((uint64_t)N << 22) |
         ((uint64_t)K << 2) | (glu ? 2u : 0u) | (kind == 1 ? 1u : 0u);
}
}  // namespace

void gemm_tuned_set(int M, int N, int K, bool glu, int kind, int nt_hint, int split) {
  std::lock_guard<std::mutex> lk(g_tuned_mu);
  g_tuned[tune_key(M, N, K, glu, kind)] = {nt_hint, split};
}
void gemm_tuned_clear() {
  std::lock_guard<std::mutex> lk(g_tuned_mu);
  g_tuned.clear();
}
bool gemm_tuned_get(int M, int N, int K, bool glu, int kind, int* nt_hint, int* split) {
  std::lock_guard<std::mutex> lk(g_tuned_mu);
  auto it = g_tuned.find(tune_key(M, N, K, glu, kind));
  if (it == g_tuned.end()) return false;
  *nt_hint = it->second.first;
  *split = it->second.second;
  return true;
}

// Plan of a bf16 product that carries no hint and no tuned plan: prompt and mixed steps of any size, models run without the
// autotuner. Leaves the hints at 0 where the older static rules below are still the better ones.
//
// M <= 64: the K-split-wave decode kernel (gemm_dec.hip) on column tiles of 16 - 64, or, for 33 - 64 rows and more than 8192 columns,
// tiles of 64 x 96 and 64 x 128, where a cost model expects the cheapest to be 1.15 times faster than the older rules (1.25 up to 16 rows; or
// just faster, from 17 rows on, where those need a second launch for their split sums and K is at most 5120, so that X in every tile
// costs little).
// A wave of 256 workgroups takes the bytes that one asks for - its weights, and X once more for every tile, which is what narrow
// products with a long K pay for - at what a CU gets, or all their weights at what the chip gets, whichever is longer. The older
// rules are priced likewise. Constants fitted over 1600 random shapes of 256 - 70000 columns and K of 256 - 16000 (11 - 12 % off on
// average, the choice 1.5 - 2.7 % above the best of all). Against the older rules: 0.68 of their time up to 16 rows, 0.84 to 32,
// 0.92 to 64: 4096 x 4096 at one row 13.6 -> 9.6 us, 32000 x 4096 at 23 rows 62 -> 48, 22016 x 4096 at 24 rows 46 -> 35 us; 512 x 11168
// SwiGLU at 32 rows (14.0 against 35.6 us) and 18368 x 816 at 17 (13.8, 21.3) stay. From 33 rows on products below 3072 columns keep
// the 64 x 64 tiles (2048 x 4096 at 64 rows: 12.2 against 14.7 us). Tiles of 96 columns are for one wave of them (22016 x 4096 SwiGLU at
// 64 rows: 53 -> 39 us); one of the two taken for every product of more than 16384 columns lost to the older rules where a second wave
// is nearly empty and where K is short (43776 x 8160 SwiGLU at 33 rows 182 -> 223 us on 128 columns, 178 on 96; 35616 x 384 at 45
// rows 10.0 -> 13.9).
//
// M > 64 and K in whole steps of 64: the cheapest of the four-wave tiles and of 256 x 256 tiles, cut or whole, by the prices below. 17 - 64 rows
// of a finished product: those tiles where they are priced below 0.97 of the older rules, or 0.86 of the decode kernel.
//
// M > 64 otherwise: the cheapest of six tiles by a cost model. A wave of the chip takes (k-steps of 64) x us per step + 5 us, an unfilled
// second workgroup per CU counts for less, a K split adds its slabs' write and read at 4.5 TB/s and a launch, and nothing
// beats the operands' bytes at 4 TB/s. Steps measured at M = 80 - 6000 over the shapes above; the choice is 2.7 % above the
// best of 60 plans on average, and 1.5 times faster than 128 x 128 tiles below 192 tiles of 256 x 256 (4096 x 4096: M = 500 56
// -> 29, M = 1000 93 -> 45, M = 1536 135 -> 66 us; 4096 x 11008 at M = 1000: 197 -> 100 us).
struct TileCost {
  int tsel;      // tile | depth code << 4 (| 512: interleaved ring)
  int bm, bn, per_cu;
  double step;   // us per 64 of k with the chip full
  double alone;  // the same with one of two workgroups per CU
};
static constexpr TileCost kTileCost[] = {
    {4, 256, 256, 1, 1.45, 1.45},           {9 | 16, 256, 128, 1, 1.02, 1.02},        {12 | 16 | 512, 128, 256, 1, 1.06, 1.06},
    {8 | 32 | 512, 128, 128, 1, 0.70, 0.70}, {11 | 32 | 512, 64, 128, 1, 0.41, 0.41}, {11 | 16, 64, 128, 2, 0.64, 0.44},
};
struct DecCost {
  // us; bytes per us and CU; a row of X against one of W; us per wave of workgroups; bytes per us; what a CU gets more beside idle ones
  double start, cu, x, wave, chip, spare;
};
static constexpr DecCost kDecCost[] = {  // up to 16, 32, 64 rows
    {2.5, 37.5e3, 0.72, 1.17, 4.58e6, 0}, {1.66, 30.4e3, 0.382, 2.37, 10.1e6, 0.231}, {1.74, 24.7e3, 0.313, 2.75, 5.32e6, 0.242}};
struct OlderCost {  // of 17 - 64 rows: us per 64 of k on tiles of 64, 128 and 256 columns; bytes per us; the same of slabs; us for their sum
  double s64, s128, s256, chip, slab, sum;
};
static constexpr OlderCost kOlderCost[] = {  // up to 32, 64 rows
    {0.334, 0.2, 1.74, 5.37e6, 2.05e6, 0.98}, {0.364, 1.04, 2.33, 4.47e6, 2.86e6, 1.07}};
struct WideCost {  // the 64-row tiles of wide products, as DecCost but for us per 64 of k
  int tsel, bn;
  double start, step, wave, chip;
};
static constexpr WideCost kWideCost[] = {{15 | 32, 96, 3.43, 0.511, 1.17, 6.19e6}, {11 | 32, 128, 0.02, 0.587, 5.44, 5.40e6}};
// waves of 256 workgroups: each takes `us` of its workgroups, and at least `read` for each of them, its share of the chip's rate
template <typename F>
static double waves_us(int wgs, double read, F us) {
  const int rest = wgs % 256;
  return (wgs >= 256 ? wgs / 256 * std::max(us(256), 256 * read) : 0.0) + (rest ? std::max(us(rest), rest * read) : 0.0);
}
static int tile_dims(int tsel, int* bm, int* bn);
static int tiles_of(int M, int N, int bm, int bn);

// 17 - 64 rows whose consumer sums the slabs: the decode kernel on 16 - 64 columns, or, from 33 rows on, 64 x 64 tiles two k-steps deep,
// whichever is priced lower together with the closing op that reads the slabs. Constants fitted over two thirds of 850 (17 - 32 rows:
// 800) random products with their add_norm behind them, N to 8192, K of 512 - 12800, weights not in the caches; the choice is 0.9 %
// (0.5 %) above the best of all on the other third. Against the plans before (tiles one step deep from 33 rows on, below 3072 columns
// without a look at the decode kernel, and K split by a rule of its length) 0.85 of the time over 1200 others, 43 of them more than 1.02,
// 1.06 at worst (54 x 6480 x 10816: 45.9 -> 48.5); a margin of 4 % beside the older plan's price would leave 13 of those and take a fifth of the
// gains back. Above 12800 in K 0.91 over 41 products (to 32 rows not measured, so that those stay with the older price), above 8192 columns
// 1.01 over 19. us with the closing op: 64 x 2048 x 2048 11.5 -> 10.5, x 4096 13.2 -> 12.6, 33 x 2048 x 4096 12.2 -> 11.7, 64 x 4096 x 4096 17.8 ->
// 16.9, 63 x 320 x 1536 11.9 -> 8.7. The layered models' closing products, 64 x 2048 x 5632 and the like, are not among them: linear_f (ops/hip.py)
// takes the plan of the finished product and leaves its slabs unsummed; this price has add_norm behind it, not their closing ops.
struct SlabCost {  // as DecCost; us of the closing op in start, slab: bytes of sums written and read per us
  double start, cu, x, wave, chip, spare, slab;
};
static constexpr SlabCost kSlabDec[] = {{4.405, 28.9e3, 0.37, 1.478, 6.19e6, 0.359, 1.57e6}, {4.442, 27.6e3, 0.341, 1.696, 5.2e6, 0.219, 1.98e6}};
static bool gemm_slab_plan(int M, int N, int K, int64_t ws_bytes, int* nt_hint, int* split) {
  if (N < 256 || N > 8192 || K < 512 || (M <= 32 && K > 12800)) return false;
  const SlabCost& c = kSlabDec[M > 32];
  const double bytes = 2.0 * N * K;
  double best = 0;
  auto take = [&](double t, int code, int s) {
    if (best == 0 || t < best) best = t, *nt_hint = code << 8, *split = s;
  };
  for (int s : {2, 4, 8}) {
    if (K / s < 256 || (int64_t)s * M * N * 4 > ws_bytes) break;
    for (int bn = 64; bn >= 16; bn -= 16) {
      const double kk = (double)K / s;
      take(c.start + s * 8.0 * M * N / c.slab + waves_us((N + bn - 1) / bn * s, kk * bn * 2 / c.chip, [&](int n) {
             return kk * (bn + c.x * M) * 2 / (c.cu * (1 + c.spare * (256 - n) / 256)) + c.wave;
           }), bn / 16 | 32 | kDecHint, s);
    }
  }
  for (int s : {2, 3, 4, 6, 8}) {
    if (M <= 32 || K / s < 128 || (int64_t)s * M * N * 4 > ws_bytes) break;
    const int per = ((K + 63) / 64 + s - 1) / s, wgs = (N + 63) / 64 * s;
    take(5.54 + s * 8.0 * M * N / 1.91e6 + std::max(std::max(per * 0.375, (wgs + 255) / 256 * per * 0.353), bytes / 5.95e6), 3 | 32, s);
  }
  return best > 0;
}

// The four-wave tiles (gemm_four.hip), from 17 rows on, by a price fitted to 60000 measurements of 14 tiles and splits of K over 7500 random
// products (17 - 8300 rows, 256 - 24000 columns, K of 256 - 12000, with and without gate or activation, weights not in the caches). The
// choice is 1.2 - 2 % above the best of all. Against the plans before, of the same products: 0.84 of the time at 33 - 48 rows, 0.80 to 64, 0.74
// to 128, 0.75 to 512, 0.76 to 1024, 0.80 to 2048, 0.84 to 4096, 0.90 above; 17 - 32 rows, where the decode kernel is mostly the better one, 0.95.
// One in a hundred takes more than 1.02 of it (one in twenty above 2048 rows); at worst 1.23 (235 x 15360 x 6400 in slabs, 72 us and 88).
// Up to 32 rows and to 128 the numbers come from 570 products of their own, K to 12800, every tile and split, plans near the best counting most: with
// those of all rows a long K was left to too few workgroups. Over 570 others 2.8 and 1.2 % above the best (3.9 and 2.4 before), up to 1.03 and 1.05 of
// the older plans (1.42 and 1.30); us, older plan, numbers of all rows, now: 25 x 5752 x 7104 22, 30, 21; 32 x 5528 x
// 11328 32, 48, 32; 121 x 10016 x 7744 48, 57, 45; 122 x 9376 x 10816 gated 58, 75, 59; 66 x 10240 x 11392 gated 54, 70, 58.
// us of a launch; of a round of workgroups, and what a gate adds; per 64 of k with one
// workgroup on a CU and with `slots` of them; how much less of that a round takes per CU left idle; the combine of split sums, once and per
// slice and 128 x 128 tile; bytes per us.
struct FourCost {
  int code, bm, bn, slots;
  double start, round, gate, alone, full, idle, sum, slice, chip;
};
static constexpr FourCost kFourFew[] = {  // up to 32 rows: weights are what there is to read
    {1, 32, 64, 2, 1.25, 2.07, 0.18, 0.389, 0.834, 0.648, 1.22, 1.19, 5.50e6}, {8, 64, 32, 2, 0.69, 2.79, 0.30, 0.228, 0.442, 0.413, 1.28, 1.64, 4.64e6},
    {13, 64, 64, 1, 0.18, 3.89, 0.40, 0.370, 0.352, 0.542, 1.45, 0.91, 10.8e6}};
static constexpr FourCost kFourMore[] = {  // up to 64 rows
    {0, 64, 64, 3, 0.00, 3.52, 0.29, 0.493, 1.411, 0.601, 1.29, 1.30, 5.36e6}, {1, 32, 64, 2, 2.16, 1.49, 0.09, 0.236, 0.512, 0.438, 1.19, 1.88, 4.10e6},
    {8, 64, 32, 2, 0.82, 2.73, 0.00, 0.224, 0.458, 0.395, 1.25, 1.88, 4.05e6}, {10, 64, 128, 2, 0.12, 3.80, 0.82, 0.833, 1.807, 0.704, 1.74, 0.85, 9.91e6},
    {13, 64, 64, 1, 0.38, 3.83, 0.31, 0.378, 0.371, 0.549, 1.33, 1.28, 13.0e6}, {12, 64, 128, 1, 0.00, 4.55, 0.79, 0.792, 0.744, 0.691, 1.79, 0.79, 4.78e6}};
static constexpr FourCost kFourMid[] = {  // up to 128 rows
    {0, 64, 64, 3, 1.10, 2.49, 0.32, 0.390, 1.010, 0.537, 1.41, 1.24, 18.1e6},  {1, 32, 64, 2, 1.33, 2.27, 0.07, 0.216, 0.428, 0.409, 1.31, 1.60, 3.32e6},
    {2, 128, 64, 2, 0.00, 3.98, 0.78, 0.577, 1.235, 0.598, 2.02, 0.81, 3.91e6}, {3, 128, 128, 2, 0.00, 3.44, 1.87, 1.299, 2.318, 0.585, 2.30, 0.74, 3.92e6},
    {4, 128, 128, 1, 0.00, 4.88, 1.73, 0.945, 0.891, 0.637, 2.16, 0.70, 4.96e6}, {6, 128, 192, 1, 0.02, 5.93, 2.29, 1.266, 1.277, 0.623, 2.34, 0.64, 4.10e6},
    {8, 64, 32, 2, 1.12, 2.56, 0.07, 0.198, 0.370, 0.348, 1.37, 1.58, 2.52e6},  {10, 64, 128, 2, 0.51, 3.53, 0.74, 0.614, 1.263, 0.621, 1.97, 0.81, 4.45e6},
    {11, 128, 64, 1, 0.00, 4.69, 0.75, 0.522, 0.455, 0.557, 1.96, 0.78, 3.70e6}, {12, 64, 128, 1, 0.00, 4.77, 0.67, 0.563, 0.483, 0.589, 1.92, 0.76, 3.73e6},
    {13, 64, 64, 1, 0.37, 4.05, 0.24, 0.289, 0.258, 0.434, 1.35, 1.27, 3.59e6}};
static constexpr FourCost kFourMany[] = {
    {0, 64, 64, 3, 3.87, 0.63, 0.23, 0.235, 0.593, 0.231, 1.72, 2.22, 2.76e6},  {1, 32, 64, 2, 2.52, 2.10, 0.03, 0.157, 0.285, 0.178, 1.61, 1.80, 13.5e6},
    {2, 128, 64, 2, 0.82, 4.36, 0.62, 0.300, 0.598, 0.257, 2.59, 1.42, 3.40e6}, {3, 128, 128, 2, 0.00, 4.75, 1.49, 0.689, 0.988, 0.342, 3.48, 1.11, 2.60e6},
    {4, 128, 128, 1, 0.00, 6.29, 1.51, 0.446, 0.454, 0.316, 3.19, 0.94, 16.3e6}, {5, 192, 128, 1, 0.00, 7.53, 1.97, 0.602, 0.633, 0.318, 3.34, 0.84, 3.41e6},
    {6, 128, 192, 1, 0.00, 7.62, 2.02, 0.617, 0.634, 0.332, 3.46, 0.81, 3.27e6}, {7, 256, 128, 1, 0.00, 8.12, 3.02, 0.781, 0.814, 0.297, 4.11, 0.82, 3.17e6},
    {8, 64, 32, 2, 2.55, 1.96, 0.00, 0.162, 0.268, 0.180, 1.63, 2.06, 19.7e6},  {9, 192, 192, 1, 0.00, 8.76, 3.23, 0.855, 0.856, 0.286, 4.34, 0.77, 3.50e6},
    {10, 64, 128, 2, 1.08, 4.24, 0.61, 0.302, 0.626, 0.236, 2.53, 1.32, 2.69e6}, {11, 128, 64, 1, 0.68, 5.01, 0.57, 0.292, 0.279, 0.225, 2.73, 1.14, 12.4e6},
    {12, 64, 128, 1, 0.80, 4.87, 0.58, 0.311, 0.299, 0.272, 2.67, 1.06, 4.76e6}, {13, 64, 64, 1, 1.74, 3.34, 0.21, 0.208, 0.192, 0.174, 2.08, 1.58, 2.28e6}};
static constexpr FourCost kQuadCost = {4, 256, 256, 1, 3.07, 5.70, 1.72, 1.465, 1.425, 0.317, 0, 0, 5.0e6};  // gemm_quad.hip
static double four_us(const FourCost& c, int M, int N, int K, bool glu, int split) {
  const int64_t wgs = (int64_t)tiles_of(M, N, c.bm, c.bn) * split, cap = 256 * c.slots, rest = wgs % cap;
  const int per = (K / 64 + split - 1) / split, held = (int)((rest + 255) / 256);
  const double round = c.round + (glu ? c.gate : 0.0);
  double t = c.start + (double)(wgs / cap) * (per * c.full + round);
  if (rest) {
    const double step = c.slots > 1 ? c.alone + (c.full - c.alone) * (held - 1) / (c.slots - 1) : c.alone;
    t += per * step * (1.0 - c.idle * (1.0 - (double)rest / (256 * held))) + round;
  }
  return std::max(t, c.start + (2.0 * N * K + 2.0 * M * K + 2.0 * M * (glu ? N / 2 : N)) / c.chip);
}
struct FourPlan {
  int hint, split;  // hint 0: none
  double us;
};
static FourPlan gemm_four_price(int M, int N, int K, bool glu, bool slabs, int64_t ws_bytes) {
  FourPlan best{0, 1, 0.0};
  auto look = [&](const FourCost& c) {
    if (glu && c.bn == 32) return;  // (a gate and its up lie in one wave)
    const int64_t tiles = tiles_of(M, N, c.bm, c.bn);
    for (int s : {1, 2, 3, 4, 6, 8}) {
      if (s > 1 && (K / s < 256 || tiles * s > 1000 || (slabs ? (int64_t)s * M * N : tiles * s * c.bm * c.bn) * 4 > ws_bytes)) break;
      if (s == 1 && slabs) continue;
      double t = four_us(c, M, N, K, glu, s);
      if (s > 1) t += slabs ? 8.0 * s * M * N / 4.5e6 : c.sum + c.slice * s * c.bm * c.bn / 16384;
      if (!best.hint || t < best.us) best = FourPlan{(c.code | kFourHint | (s > 1 && !slabs ? 256 : 0)) << 8, s, t};
    }
  };
  if (M <= 32) {
    for (const FourCost& c : kFourFew) look(c);
  } else if (M <= 64) {
    for (const FourCost& c : kFourMore) look(c);
  } else if (M <= 128) {
    for (const FourCost& c : kFourMid) look(c);
  } else {
    for (const FourCost& c : kFourMany) look(c);
  }
  return best;
}

// A thread's last answers by size, which depend on nothing else: 64 sets of four, of which the oldest makes room. 40 - 84 prices take 0.5 - 0.9 us and a
// cut 1 - 3, and a product is planned two or three times, more than the launch that it is for leaves where a step of few rows waits for the host.
// (64 single places, by the exclusive or of three products: two sizes met at every number of rows or at none, GPT-2 XL's 4800 x 1600 and 6400 x 1600 at
// every one, so that its four sizes in turn took 0.77 us a plan, now 0.32; 8260 x 10240 x 2048 with its cut 2.7, now 0.41.)
static thread_local int64_t g_priced = 0;
int64_t gemm_priced() { return g_priced; }
template <typename V>
struct BySize {
  struct Entry {
    int M, N, K, kind;
    int64_t ws;
    V value;
  };
  Entry of[64][4] = {};
  uint8_t oldest[64] = {};
  template <typename F>
  V get(int M, int N, int K, int kind, int64_t ws, F make) {
    uint32_t h = (uint32_t)M * 0x9e3779b1u;
    h = (h ^ h >> 15 ^ (uint32_t)N) * 0x85ebca6bu;
    h = (h ^ h >> 15 ^ (uint32_t)K << 2 ^ (uint32_t)kind) * 0xc2b2ae35u;
    h >>= 26;
    for (const Entry& e : of[h])
      if (e.M == M && e.N == N && e.K == K && e.kind == kind && e.ws == ws) return e.value;
    ++g_priced;
    const V value = make();
    of[h][oldest[h]++ & 3] = Entry{M, N, K, kind, ws, value};
    return value;
  }
};

// slabs: split sums are left to the consumer
static FourPlan gemm_four_plan(int M, int N, int K, bool glu, bool slabs, int64_t ws_bytes) {
  if (M < 17 || N % 8 || K % 64) return FourPlan{0, 1, 0.0};
  static thread_local BySize<FourPlan> kept;
  return kept.get(M, N, K, glu | slabs << 1, ws_bytes, [&] { return gemm_four_price(M, N, K, glu, slabs, ws_bytes); });
}

// slabs: the consumer sums split-K slabs itself and so gets the product in 32 bits. Where the older rules split K that stays so:
// only split plans are looked at, their slabs costing a write and a read and no launch.
static double quad_us(int M, int N, int K, bool glu, int64_t ws_bytes);
static void gemm_static_plan(int M, int N, int K, bool glu, bool slabs, int64_t ws_bytes, int* nt_hint, int* split, bool four = true) {
  if (N % 8 || K % 16) return;
  if (slabs) {
    int t = 0, s = 0;
    if (M <= 16) gemm_stream_plan(M, N, K, &t, &s);
    else gemm_tiled_plan(M, N, K, &t, &s, glu);
    slabs = s > 1 && (int64_t)s * M * N * 4 <= ws_bytes;
  }
  if (M <= 64) {
    if (slabs && M > 16 && gemm_slab_plan(M, N, K, ws_bytes, nt_hint, split)) return;
    const double bytes = 2.0 * N * K, slab = 8.0 * M * N / 2.5e6;
    double older, faster = M <= 16 ? 1.25 : 1.15;
    if (M <= 16) {
      int nt, s;
      gemm_stream_plan(M, N, K, &nt, &s);
      older = 2.0 + std::max(((K + 255) / 256 + s - 1) / s * 2.17 * nt, bytes / 3.03e6) + (s > 1 && !slabs ? 2.9 : 0.0);
    } else {
      const OlderCost& c = kOlderCost[M > 32];
      int t = 0, s = 0, bm, bn;
      gemm_tiled_plan(M, N, K, &t, &s, glu);
      tile_dims(t & 15, &bm, &bn);
      const double step = (t & 15) == 4 ? c.s256 : (bn == 64 ? c.s64 : c.s128);
      older = 4.71 + std::max(((K + 63) / 64 + s - 1) / s * step, bytes / c.chip);
      if (s > 1) older += s * 8.0 * M * N / c.slab + (slabs ? 0.0 : c.sum);
      if (s > 1 && !slabs && K <= 5120) faster = 1.0;  // (else two launches, the second waiting for the first)
    }
    // gated products take the older kernels longer than their plain ones of the same size: 12 x 17472 x 3488 63 us, on the decode kernel 38, 61 x
    // 18688 x 4656 78, on tiles of 96 columns 58
    if (glu) older *= M <= 16 ? 1.4 : 1.15;
    const DecCost& c = kDecCost[M <= 16 ? 0 : M <= 32 ? 1 : 2];
    double best = 0;
    int code = 0, sp = 1;
    for (int s = slabs ? 2 : 1; s <= (slabs ? 4 : 1); s *= 2) {
      if (M > 32 && N < 3072) break;
      if (s > 1 && (K / s < 256 || (int64_t)s * M * N * 4 > ws_bytes)) break;
      for (int bn = 64; bn >= 16; bn -= 16) {
        if (glu && bn % 32) continue;
        const double t = c.start + (s > 1 ? s * slab : 0.0) +
                         waves_us((N + bn - 1) / bn * s, (double)K / s * bn * 2 / c.chip, [&](int n) {
                           return (double)K / s * (bn + c.x * M) * 2 / (c.cu * (1 + c.spare * (256 - n) / 256)) + c.wave;
                         });
        if (!code || t < best) best = t, code = bn / 16 | 32 | 1024, sp = s;
      }
    }
    if (M > 32 && N > 8192 && !slabs) {
      for (const WideCost& w : kWideCost) {
        const double t = w.start + waves_us((N + w.bn - 1) / w.bn, 2.0 * K * w.bn / w.chip,
                                            [&](int) { return (K + 63) / 64 * w.step + w.wave; });
        if (t < best) best = t, code = w.tsel;
      }
    }
    const bool dec = code && best * faster <= older;
    if (dec) *nt_hint = code << 8, *split = sp;
    if (!four || slabs) return;
    const FourPlan p = gemm_four_plan(M, N, K, glu, false, ws_bytes);
    if (p.hint && p.us < (dec ? 0.86 * best : 0.97 * older)) *nt_hint = p.hint, *split = p.split;
    return;
  }
  const FourPlan p = gemm_four_plan(M, N, K, glu, slabs, ws_bytes);
  if (p.hint) {
    const bool quad = !slabs && quad_us(M, N, K, glu, ws_bytes) <= p.us;
    *nt_hint = quad ? 4 << 8 : p.hint;
    *split = quad ? 1 : p.split;
    return;
  }
  // two rows of 64 x 64 tiles, two to three workgroups per CU: the older rule's one launch of them is the faster one until K is long
  // (22016 x 2656 at 80 rows: 42.7 against 47.4 us; x 4096: 53.6 and 54.4; 16640 x 5120: 57.5 and 52.9)
  const int t64 = tiles_of(M, N, 64, 64);
  if (glu && M <= 128 && t64 > 512 && t64 <= 768 && K < 3900) return;
  const int nk = (K + 63) / 64;
  const double bytes = 2.0 * N * K + 2.0 * M * K + 2.0 * M * (glu ? N / 2 : N);
  double best = 0;
  for (const TileCost& c : kTileCost) {
    for (int s : {1, 2, 3, 4, 6, 8}) {
      if (s == 1 && slabs) continue;
      if (s > 1 && (c.tsel == 4 || K / s < 256 || (int64_t)s * M * N * 4 > ws_bytes)) break;
      const int per = (nk + s - 1) / s;
      const int64_t wgs = (int64_t)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * s, slots = 256 * c.per_cu;
      const int64_t rest = wgs % slots;
      double t = (double)(wgs / slots) * (per * c.step + 5.0);
      if (rest) t += per * (rest <= 256 ? c.alone : c.step) + 5.0;
      t = std::max(t, bytes / 4.0e6);
      if (s > 1) t += (slabs ? 0.0 : 4.0) + 8.0 * s * M * N / 4.5e6;
      if (best == 0 || t < best) {
        best = t;
        *nt_hint = (K % 64 ? c.tsel & ~512 : c.tsel) << 8;
        *split = s;
      }
    }
  }
}

// The same for fp8 weights and up to 32 rows: the decode kernel, priced as above (constants fitted over 420 random shapes of 512 - 60000
// columns and K of 256 - 16000: 5 - 7 % off on average, its choice of columns and split 0.3 % above the best), instead of the
// streaming kernel (up to 16 rows) and the 64 x 64 tiles. 0.72 of their time on average: us at 23 rows, 12288 x 4096 24.8 -> 13.7,
// 22016 x 4096 SwiGLU 39.0 -> 27.6, slabs of 4096 x 11008 18.4 -> 12.6 and of 4096 x 4096 10.0 -> 6.7; at one row 16.1 -> 12.3,
// 26.3 -> 23.3, 14.3 -> 10.7, 7.2 -> 5.7. The older rules stay where they are faster: many waves of a short K (53344 x 256 at one row
// 6.7 against 13.6, 57056 x 576 SwiGLU 12.3 and 19.4), and SwiGLU of few columns and a long K, which they split (1856 x 12240 at 15 rows 18.3
// and 23.6; but 1888 x 6528 at 13 rows 0.63 the other way, where the line lies between).
struct DecF8Cost {  // as DecCost; slab: bytes of split sums written and read per us, sum: us of their launch
  double start, cu, x, wave, chip, spare, slab, sum;
};
static constexpr DecF8Cost kDecF8Cost[] = {{1.82, 22.3e3, 0.644, 2.05, 4.99e6, 0.415, 100e6, 1.63},
                                           {1.98, 20.1e3, 0.582, 1.93, 4.38e6, 0.376, 3.94e6, 1.94}};
static void gemm_static_plan_f8(int M, int N, int K, bool glu, bool slabs, int64_t ws_bytes, int* nt_hint, int* split) {
  if (M > 32 || N % 8 || K % 16) return;
  if ((N > 16384 && K < 1024) || (N > 8192 && K < 512) || (glu && N <= 2816 && K >= 6000)) return;
  if (slabs) {
    int t = 0, s = 0;
    if (M <= 16) gemm_stream_plan(M, N, K, &t, &s);
    else gemm_tiled_plan(M, N, K, &t, &s, glu);
    slabs = s > 1 && (int64_t)s * M * N * 4 <= ws_bytes;
  }
  const DecF8Cost& c = kDecF8Cost[M > 16];
  const int k = (K + 127) / 128 * 128;
  double best = 0;
  int code = 0, sp = 1;
  for (int s = slabs ? 2 : 1; s <= (glu ? 1 : 8); s *= 2) {
    if (s > 1 && (K / s < 512 || (int64_t)s * M * N * 4 > ws_bytes)) break;
    for (int bn = 64; bn >= 16; bn -= 16) {
      if (glu && bn % 32) continue;
      const double kk = (double)k / s;
      double t = c.start + waves_us((N + bn - 1) / bn * s, kk * bn / c.chip, [&](int n) {
                   return kk * (bn + c.x * M) / (c.cu * (1 + c.spare * (256 - n) / 256)) + c.wave;
                 });
      if (s > 1) t += s * 4.0 * M * N / c.slab + (slabs ? 0.0 : c.sum);
      if (!code || t < best) best = t, code = bn / 16 | 32 | kDecHint, sp = s;
    }
  }
  if (!code) return;
  *nt_hint = code << 8;
  *split = sp;
}

// Operands that every tile of gemm_static_plan takes: rows of 16-byte alignment, 256 of them within a descriptor of 31 bits
// (strides below 4.2 M numbers). Anything else keeps the older rules.
static bool gemm_static_takes(bool w_fp8, const void* x, int64_t ldx, const void* w, int64_t ldw) {
  return ldx % 8 == 0 && ldw % (w_fp8 ? 16 : 8) == 0 && !(((uintptr_t)x | (uintptr_t)w) & 15) && std::max(ldx, ldw) < (1 << 22);
}

// The plan of a product: its hints, else a tuned plan, else the static one where it applies. Hints of 0 remain where the older
// rules choose.
static void gemm_default_plan(int M, int N, int K, bool w_fp8, bool glu, bool slabs, int64_t ws_bytes, bool takes, int* nt_hint,
                              int* split) {
  if (*nt_hint || *split || gemm_tuned_get(M, N, K, glu, w_fp8 ? 1 : 0, nt_hint, split)) return;
  if (takes && w_fp8) gemm_static_plan_f8(M, N, K, glu, slabs, ws_bytes, nt_hint, split);
  else if (takes) gemm_static_plan(M, N, K, glu, slabs, ws_bytes, nt_hint, split);
}
static int slabs_of_plan(int M, int N, int K, bool w_fp8, bool glu, int act, int nt_hint, int split_hint, int64_t ws_bytes);

// Where to cut a product of 256 x 256 tiles whose last wave is mostly empty in two launches: the tiles of whole waves, and the rows or
// columns left over, which smaller tiles spread over the chip. What the launches run with is gemm_rest_plan's; where the cut lies is priced with
// numbers of the kernels before them (kTileCost; waves that are at most 0.8 full cost only 0.78: the clock rises as tiles end; up to 64 rows left over
// read all weights at 4.5 TB/s behind 8 us), and those places still hold: over 204 random products that it cuts, 257 - 10000 rows and whole steps of
// k, two launches take 0.888 of the time of one, 1.03 at worst, two of them above 1.02 (K from 1024 on 0.869, 1.01 at worst; below 0.934). us, one
// launch and two: 1773 x 12288 x 4096 186 and 157, SwiGLU x 22016 277 and 263, 8261 x 2048 x 2048 86 and 61, x 4096 163 and 108, 8261 x 6400 x 2048
// 192 and 179, 3999 x 22016 x 4096 561 and 541. Left whole: 8192 x 5120 x 2048 (2.5 waves) 145, 8192 x 9472 x 2048 (4.6) 249, 5000 x 12288 x 4096
// (3.75) 373.
// Below K = 1024 a tile's start and end are half of it, and what is promised up to there does not come: ungated products are cut there where more than
// 6.5 % are promised, others from 3 % on.
// The rest's tiles can be too few for the chip (69 x 2048): a split of K, priced a tenth below the best of the tiles looked at before, up to 24 MB of
// sums, lets the cut lie elsewhere, but not where that would leave up to 64 rows, whose price is too high (4106 x 15840 x 11520, ten rows left or 480
// columns 1110 and 1180 us). 1240 x 13248 x 3392 140 us in one launch and 104 in two, 2579 x 7120 x 8576 335 and 262.
struct GemmCut {
  int rows, cols;  // of the first launch; 0: not cut
};
static GemmCut gemm_cut_place(int M, int N, int K, bool glu, int64_t ws_bytes) {
  const int ntm = (M + 255) / 256, ntn = (N + 255) / 256, nk = (K + 63) / 64;
  auto tiles_us = [&](const TileCost& c, int m, int n, int split = 1) {
    const int slots = 256 * c.per_cu, wgs = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * split, rest = wgs % slots;
    const int per = (nk + split - 1) / split;
    double t = wgs / slots * (per * c.step + 5.0);
    if (rest) t += (per * (rest <= 256 ? c.alone : c.step) + 5.0) * (rest * 5 <= slots * 4 ? 0.78 : 1.0);
    t = std::max(t, (2.0 * n * K + 2.0 * m * K + 2.0 * m * (glu ? n / 2 : n)) / 4.0e6);
    return split > 1 ? t + 4.0 + 8.0 * split * m * n / 4.5e6 : t;
  };
  GemmCut cut{0, 0};
  bool few = false;  // (up to 64 rows left over)
  double best = (K < 1024 && !glu ? 0.935 : 0.97) * tiles_us(kTileCost[0], M, N);
  auto consider = [&](int rows, int cols, bool splits) {
    if (rows <= 0 || cols <= 0 || (rows >= M && cols >= N)) return;
    const int last = (rows < M ? rows / 256 * ntn : ntm * (cols / 256)) % 256;
    if (last && last < 218) return;  // whole waves, the last of them at least 0.85 full
    const int m = rows < M ? M - rows : M, n = cols < N ? N - cols : N;
    double rest = 8.0 + 2.0 * n * K / 4.5e6;
    int split = 0;
    for (const TileCost& c : kTileCost) {
      if (m <= 64) break;
      for (int s : {1, 2, 3, 4, 6, 8}) {
        if (s > 1 && (!splits || c.tsel == 4 || K / s < 256 || (int64_t)s * m * n * 4 > std::min<int64_t>(ws_bytes, 24 << 20))) break;
        const double t = tiles_us(c, m, n, s);
        if (!split || t < (s > split ? 0.9 : 1.0) * rest) rest = t, split = s;
      }
    }
    const double t = tiles_us(kTileCost[0], std::min(rows, M), std::min(cols, N)) + rest;
    if (t < best) best = t, few = m <= 64, cut = GemmCut{rows < M ? rows : 0, cols < N ? cols : 0};
  };
  const int waves = (int)std::min<int64_t>((int64_t)ntm * ntn / 256, 64);
  for (bool splits : {false, true}) {
    for (int w = 1; w <= waves; ++w) {
      consider(256 * w / ntn * 256, N, splits);
      consider(M, 256 * w / ntm * 256, splits);
    }
    consider((ntm - 1) * 256, N, splits);
    if (cut.rows && few) break;
  }
  return cut;
}

static GemmCut gemm_cut(int M, int N, int K, bool glu, int64_t ws_bytes) {
  static thread_local BySize<GemmCut> kept;
  return kept.get(M, N, K, glu, ws_bytes, [&] { return gemm_cut_place(M, N, K, glu, ws_bytes); });
}

// What the second launch runs with: four-wave tiles from 65 rows on, else the plan of its size (hint 0)
static FourPlan gemm_rest_plan(int m, int n, int K, bool glu, int64_t ws_bytes) {
  const FourPlan p = m > 64 ? gemm_four_plan(m, n, K, glu, false, ws_bytes) : FourPlan{0, 0, 0.0};
  return p.hint ? p : FourPlan{0, 0, 8.0 + 2.0 * n * K / 4.5e6};
}

// 256 x 256 tiles, cut or whole
static double quad_us(int M, int N, int K, bool glu, int64_t ws_bytes) {
  const GemmCut cut = gemm_cut(M, N, K, glu, ws_bytes);
  if (!cut.rows && !cut.cols) return four_us(kQuadCost, M, N, K, glu, 1);
  const int rows = cut.rows ? cut.rows : M, cols = cut.cols ? cut.cols : N;
  return four_us(kQuadCost, rows, cols, K, glu, 1) + gemm_rest_plan(rows < M ? M - rows : M, cols < N ? N - cols : N, K, glu, ws_bytes).us;
}

int launch_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, bool w_fp8, const void* w_scale,
                const void* bias, void* y, int64_t ldy, int M, int N, int K, int act, bool glu, void* workspace,
                int64_t ws_bytes, int nt_hint, int split_hint, bool partial_out, hipStream_t st) {
  if (M == 0 || N == 0) return 0;
  int tuned_nt, tuned_split;
  const bool free_plan = !nt_hint && !split_hint && !w_fp8 && !gemm_tuned_get(M, N, K, glu, 0, &tuned_nt, &tuned_split);
  gemm_default_plan(M, N, K, w_fp8, glu, partial_out && !glu && act == 0, ws_bytes, gemm_static_takes(w_fp8, x, ldx, w, ldw), &nt_hint,
                    &split_hint);
  if (free_plan && nt_hint == 4 << 8 && y && !(glu && N % 32) && gemm_quad_ok(N, K, ldx, ldw, 256, y, ldy, 2, glu)) {
    const GemmCut cut = gemm_cut(M, N, K, glu, ws_bytes);
    if (cut.rows) {
      launch_gemm(x, ldx, w, ldw, false, nullptr, bias, y, ldy, cut.rows, N, K, act, glu, workspace, ws_bytes, 4 << 8, 1, false, st);
      const FourPlan rest = gemm_rest_plan(M - cut.rows, N, K, glu, ws_bytes);
      return launch_gemm((const bf16_t*)x + cut.rows * ldx, ldx, w, ldw, false, nullptr, bias, (bf16_t*)y + cut.rows * ldy, ldy,
                         M - cut.rows, N, K, act, glu, workspace, ws_bytes, rest.hint, rest.split, false, st);
    }
    if (cut.cols) {
      launch_gemm(x, ldx, w, ldw, false, nullptr, bias, y, ldy, M, cut.cols, K, act, glu, workspace, ws_bytes, 4 << 8, 1, false, st);
      const FourPlan rest = gemm_rest_plan(M, N - cut.cols, K, glu, ws_bytes);
      return launch_gemm(x, ldx, (const bf16_t*)w + cut.cols * ldw, ldw, false, nullptr, bias ? (const bf16_t*)bias + cut.cols : nullptr,
                         (bf16_t*)y + (glu ? cut.cols / 2 : cut.cols), ldy, M, N - cut.cols, K, act, glu, workspace, ws_bytes, rest.hint,
                         rest.split, false, st);
    }
  }
  if (!y && (!partial_out || slabs_of_plan(M, N, K, w_fp8, glu, act, nt_hint, split_hint, ws_bytes) == 0))
    throw std::runtime_error("gemm: this configuration writes the output, but no output buffer was given");
  if (K % 16) throw std::runtime_error("gemm: K must be a multiple of 16");
  if (glu && (N % 32)) throw std::runtime_error("gemm: glu needs N % 32 == 0");
  auto X = (const bf16_t*)x;
  auto B = (const bf16_t*)bias;
  auto Y = (bf16_t*)y;
  auto WS = (const float*)w_scale;
  const int g = glu ? 1 : 0;
  // weight-streaming kernel: M <= 16, explicit stream hints, and fp8 prefill panels; fp8 decode
  // (16 < M <= 128) runs the tiled kernel with fp8 weight tiles (W8A16)
  const int tiled_hint = nt_hint >> 8;
  const bool stream = (nt_hint & 0xff) || (!tiled_hint && (M <= 16 || (w_fp8 && M > 128)));
  if (stream) {
    if (M > 128) {  // fp8 weights with many rows (prefill): 128-row panels through the streaming kernel
      for (int m0 = 0; m0 < M; m0 += 128) {
        const int mm = std::min(128, M - m0);
        launch_gemm((const bf16_t*)x + m0 * ldx, ldx, w, ldw, w_fp8, w_scale, bias, (bf16_t*)y + m0 * ldy, ldy, mm, N,
                    K, act, glu, workspace, ws_bytes, nt_hint, split_hint, false, st);
      }
      return 0;
    }
    int nt, splitk;
    gemm_stream_plan(M, N, K, &nt, &splitk);
    // nt_hint = nt + 16 * variant (variant 1: LDS-DMA X staging, 2: register-staged X + W ring)
    int variant = ((nt_hint >> 4) & 15) ? ((nt_hint >> 4) & 15) : 2;
    nt_hint &= 15;
    if (nt_hint > 0) nt = nt_hint;
    if (split_hint > 0) splitk = split_hint;
    if (glu && nt < 2) nt = 2;  // the SwiGLU epilogue pairs (gate, up) 16-column tiles inside a wave
    if ((int64_t)splitk * M * N * 4 > ws_bytes) splitk = 1;
    float* part = splitk > 1 ? (float*)workspace : nullptr;
    const int mt = (M + 15) / 16;
    const int act_k = splitk > 1 ? 0 : act, glu_k = splitk > 1 ? 0 : g;
    if (w_fp8) launch_stream<true>(variant, mt, nt, X, ldx, w, ldw, WS, B, Y, ldy, part, M, N, K, act_k, glu_k, splitk, st);
    else launch_stream<false>(variant, mt, nt, X, ldx, w, ldw, nullptr, B, Y, ldy, part, M, N, K, act_k, glu_k, splitk, st);
    if (splitk > 1 && partial_out && !glu && act == 0) return splitk;
    if (splitk > 1) {
      const int nout = glu ? N / 2 : N;
      dim3 grid(std::min((nout + 255) / 256, 64), M);
      splitk_reduce_kernel<<<grid, 256, 0, st>>>(part, splitk, M, N, B, Y, ldy, act, g);
      HIP_CHECK_LAUNCH();
    }
    return 0;
  }
  return launch_tiled(X, ldx, w, ldw, B, Y, ldy, M, N, K, act, g, nt_hint >> 8, split_hint, workspace,
                      ws_bytes, partial_out, st, w_fp8 ? WS : nullptr);
}

// Tiled-path plan. Tile: 64 rows for M <= 64 (64x64, or 64x128 when 64x64 gives > 256 tiles),
// else 128x128. K is split until the grid holds ~3 (64-row tiles) or ~1.5 (128x128) workgroups
// per CU, keeping >= 512 k per slice. Measured on the Llama-2-7B shapes at M = 64..512
// (bench/gemm_bench.py --sweep): within ~5% of the best (tile, split) of the sweep everywhere.
static int tiles_of(int M, int N, int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); }
// tsel: 1 = 128x128, 2 = 64x128, 3 = 64x64 (4 waves); 5 = 256x128, 6 = 256x64 (8 waves, 1 WG/CU);
// 4 = the big-tile kernel
bool gemm_mid_dims(int tsel, int* bm, int* bn, int* threads);

// tsel 8-12: gemm_mid (gemm_mid.hip: buffer-descriptor staging, 128x128 / 256x128 / 64x256 / 64x128 / 128x256)
static int tile_dims(int tsel, int* bm, int* bn) {
  int thr;
  if (gemm_mid_dims(tsel, bm, bn, &thr)) return 0;
  *bm = tsel >= 5 ? 256 : (tsel == 1 ? 128 : 64);
  *bn = (tsel == 3 || tsel == 6) ? 64 : 128;
  return 0;
}
void gemm_tiled_plan(int M, int N, int K, int* tsel_io, int* split_io, bool glu) {
  int tsel = *tsel_io;
  // SwiGLU output cannot be folded into the next kernel, so a split would cost its own reduce
  // launch: with >= 256 64x64 tiles, no split (measured equal or better at M <= 128)
  if (tsel == 0 && glu && M <= 128 && tiles_of(M, N, 64, 64) >= 256 && *split_io <= 0) {
    *tsel_io = 3 | 16;
    *split_io = 1;
    return;
  }
  if (tsel == 0) {
    if (tiles_of(M, N, 256, 256) >= 192) tsel = 4;
    else tsel = M <= 64 ? (tiles_of(M, N, 64, 64) > 256 ? 2 : 3) : 1;
  }
  int hint_bits = tsel & ~15;
  tsel &= 15;
  if (tsel >= 5) hint_bits &= ~128;  // no stream-K variant of the 8-wave tiles
  if (hint_bits & 128) {  // stream-K: output is final (no slabs); split_io carries workgroups per CU
    *tsel_io = tsel | hint_bits;
    if (*split_io <= 0) *split_io = 2;
    return;
  }
  if (tsel == 4) {  // big-tile kernel: no split-K, no stage option
    *tsel_io = 4;
    *split_io = 1;
    return;
  }
  int bm, bn;
  tile_dims(tsel, &bm, &bn);
  const int nt = tiles_of(M, N, bm, bn);
  int s = *split_io;
  if (s <= 0) {
    const int bound = bm == 64 ? 800 : (bm == 128 ? 537 : 300);
    s = 1;
    while (nt * s * 2 <= bound && s < 8 && K / (2 * s) >= 512) s *= 2;
  }
  s = std::max(1, std::min(s, (K + TBK - 1) / TBK));
  // 3-stage LDS ring when the grid is too small for block-level latency hiding (measured: o/down
  // projections and the LM head at M <= 128 gain 10-20%; wide grids lose occupancy to its LDS)
  if (*tsel_io == 0 && nt * s <= (bm == 64 ? 600 : 256)) tsel |= 16;
  *tsel_io = tsel | hint_bits;
  *split_io = s;
}

static bool wnt_ok(int tsel_raw, int M, int tsel) {
  int bm, bn;
  tile_dims(tsel & 15, &bm, &bn);
  return !(tsel_raw & 64) && M <= bm;
}

// per-tile arrival counters of the stream-K and split-K combines, one buffer per device: zeroed
// once, reset by every last arriver (consecutive GEMMs on one stream never overlap)
static std::mutex g_sk_mu;
static int* g_sk_counters[64] = {};
static int g_sk_capacity[64] = {};

// workspace slot (gemm_set_slot): GEMM chains that may run concurrently on different streams (the two
// half-batch decode chains, models/decoder.py) use disjoint counter ranges, as they use disjoint workspaces
static constexpr int kSlots = 4;
static thread_local int g_ws_slot = 0;
void gemm_set_slot(int s) { g_ws_slot = s & (kSlots - 1); }

// `on`: the stream of a launch by its own rules. Where it is being captured and the counters are not there yet, null is returned; else they are made
// on it, so that another thread's capture is not disturbed (an allocation under the strict mode, or a wait for the device, would end it).
static int* sk_counters(int n, const hipStream_t* on = nullptr) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) throw std::runtime_error("gemm counters: bad device");
  std::lock_guard<std::mutex> lk(g_sk_mu);
  if (n <= g_sk_capacity[dev]) return g_sk_counters[dev] + (size_t)g_ws_slot * g_sk_capacity[dev];
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  int cap = std::max(n, 1 << 16);
  int* p = nullptr;
  const size_t bytes = (size_t)cap * kSlots * sizeof(int);
  if (on) {
    (void)hipStreamIsCapturing(*on, &cs);
    if (cs != hipStreamCaptureStatusNone) return nullptr;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const bool made = hipMalloc(&p, bytes) == hipSuccess && hipMemsetAsync(p, 0, bytes, *on) == hipSuccess &&
                      hipStreamSynchronize(*on) == hipSuccess;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (!made) throw std::runtime_error("gemm counters: not allocated");
  } else {
    (void)hipStreamIsCapturing(nullptr, &cs);
    if (cs != hipStreamCaptureStatusNone) throw std::runtime_error("gemm counters must be allocated before capture");
    if (hipMalloc(&p, bytes) != hipSuccess) throw std::runtime_error("gemm counters: hipMalloc");
    if (hipMemset(p, 0, bytes) != hipSuccess) throw std::runtime_error("gemm counters: memset");
    (void)hipDeviceSynchronize();
  }
  g_sk_counters[dev] = p;  // the old (smaller) buffer is left to the process: launches may still reference it
  g_sk_capacity[dev] = cap;
  return p + (size_t)g_ws_slot * cap;
}

// 4 KiB of zeros per device: the source of the chunks past K in gemm_pp's partial last K-tile
static const char* g_zero_page[64] = {};
static const char* zero_page() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) throw std::runtime_error("gemm zero page: bad device");
  std::lock_guard<std::mutex> lk(g_sk_mu);
  if (g_zero_page[dev]) return g_zero_page[dev];
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  (void)hipStreamIsCapturing(nullptr, &cs);
  if (cs != hipStreamCaptureStatusNone) throw std::runtime_error("gemm zero page must be allocated before capture");
  char* p = nullptr;
  if (hipMalloc(&p, 4096) != hipSuccess) throw std::runtime_error("gemm zero page: hipMalloc");
  if (hipMemset(p, 0, 4096) != hipSuccess) throw std::runtime_error("gemm zero page: memset");
  (void)hipDeviceSynchronize();
  g_zero_page[dev] = p;
  return p;
}

void gemm_reserve_streamk(int n) {
  sk_counters(n);
  (void)zero_page();
}

static bool launch_streamk(const bf16_t* X, int64_t ldx, const bf16_t* W, int64_t ldw, const bf16_t* B, bf16_t* Y,
                           int64_t ldy, int M, int N, int K, int act, int g, int tsel, int ns, int per_cu,
                           void* workspace, int64_t ws_bytes, bool wnt, hipStream_t st) {
  int bm, bn;
  tile_dims(tsel, &bm, &bn);
  if (tsel == 1 && ns > 3) ns = 3;
  if (tsel == 2 && ns > 4) ns = 4;
  if (ns == 6) ns = 4;
  const int tiles = tiles_of(M, N, bm, bn), nk = (K + TBK - 1) / TBK;
  const int64_t U = (int64_t)tiles * nk;
  if (U >= (1LL << 31)) return false;
  const int G = (int)std::min<int64_t>(U, 256LL * std::max(1, std::min(per_cu, 8)));
  const int64_t per = U / G;  // >= 1
  const int maxseg = (int)std::min<int64_t>(G, (nk + per - 1) / per + 1);
  if ((int64_t)tiles * maxseg * bm * bn * 4 > ws_bytes) return false;
  int* cnt = sk_counters(tiles);
  float* part = (float*)workspace;
#define SK(BM_, BN_, NS_)                                                                                          \
  do {                                                                                                             \
    if (wnt)                                                                                                       \
      gemm_streamk_kernel<BM_, BN_, NS_, true><<<G, 256, 0, st>>>(X, ldx, W, ldw, B, Y, ldy, part, cnt, maxseg, M, N, \
                                                                   K, act, g);                                     \
    else                                                                                                           \
      gemm_streamk_kernel<BM_, BN_, NS_, false><<<G, 256, 0, st>>>(X, ldx, W, ldw, B, Y, ldy, part, cnt, maxseg, M, \
                                                                    N, K, act, g);                                 \
  } while (0)
  if (tsel == 1) {
    if (ns == 3) SK(128, 128, 3); else SK(128, 128, 2);
  } else if (tsel == 2) {
    if (ns == 4) SK(64, 128, 4); else if (ns == 3) SK(64, 128, 3); else SK(64, 128, 2);
  } else {
    if (ns == 4) SK(64, 64, 4); else if (ns == 3) SK(64, 64, 3); else SK(64, 64, 2);
  }
#undef SK
  HIP_CHECK_LAUNCH();
  return true;
}

int launch_tiled(const bf16_t* X, int64_t ldx, const void* W, int64_t ldw, const bf16_t* B, bf16_t* Y, int64_t ldy,
                 int M, int N, int K, int act, int g, int tsel, int split_hint, void* workspace, int64_t ws_bytes,
                 bool partial_out, hipStream_t st, const float* wscale, const QkvEpi* qe) {
  const QkvEpi qv = qe ? *qe : QkvEpi{};
  const int tsel_raw = tsel;
  int s = split_hint;
  const bool f8 = wscale != nullptr;  // fp8-e4m3 weights (W8A16): half the weight bytes of a decode step
  if (tsel & kDecHint) {  // K split over the waves (gemm_dec.hip), M <= 64
    s = dec_split(M, N, K, split_hint, ws_bytes);
    if (s > 1 && Y && dec_combine_fits(N, tsel, s, ws_bytes)) {  // split-K combined in the launch: finished Y
      int bn;
      gemm_dec_bn(tsel & 15, &bn);
      static constexpr int kDecDepthC[4] = {2, 3, 4, 4};
      launch_gemm_dec(tsel & 15, kDecDepthC[(tsel >> 4) & 3], X, ldx, W, ldw, wscale, B, Y, ldy,
                      (float*)workspace, M, N, K, act, g, s, st, qe, sk_counters((N + bn - 1) / bn));
      return 0;
    }
    if (qe && s > 1) throw std::runtime_error("gemm_dec: the QKV epilogue needs an unsplit or in-launch-combined plan");
    static constexpr int kDecDepth[4] = {2, 3, 4, 4};
    float* part = s > 1 ? (float*)workspace : nullptr;
    launch_gemm_dec(tsel & 15, kDecDepth[(tsel >> 4) & 3], X, ldx, W, ldw, wscale, B, Y, ldy, part, M, N, K,
                    s > 1 ? 0 : act, s > 1 ? 0 : g, s, st, qe, nullptr);
    if (s > 1 && partial_out && !g && act == 0) return s;
    if (s > 1) {
      const int nout = g ? N / 2 : N;
      dim3 rgrid(std::min((nout + 255) / 256, 64), M);
      splitk_reduce_kernel<<<rgrid, 256, 0, st>>>(part, s, M, N, B, Y, ldy, act, g);
      HIP_CHECK_LAUNCH();
    }
    return 0;
  }
  if ((tsel & kFourHint) && (f8 || !gemm_four_ok(N, K, ldx, ldw, Y, ldy, g != 0))) tsel = split_hint = s = 0;
  if (tsel & kFourHint) {  // tiles by four waves (gemm_four.hip)
    int bm, bn;
    if (!gemm_four_dims(tsel & 15, &bm, &bn)) throw std::runtime_error("gemm: no such tile");
    const int nt = tiles_of(M, N, bm, bn);
    s = std::max(1, split_hint);
    int* cnt = (tsel & 256) && s > 1 && Y && (int64_t)nt * s * bm * bn * 4 <= ws_bytes ? sk_counters(nt, &st) : nullptr;
    if (!cnt && (qe || (int64_t)s * M * N * 4 > ws_bytes)) s = 1;
    const bool slabs = s > 1 && !cnt;
    launch_gemm_four(tsel & 15, X, ldx, (const bf16_t*)W, ldw, B, Y, ldy, s > 1 ? (float*)workspace : nullptr, M, N, K, slabs ? 0 : act,
                     slabs ? 0 : g, s, 4, st, cnt, qe);
    if (!slabs || (partial_out && !g && act == 0)) return slabs ? s : 0;
    const int nout = g ? N / 2 : N;
    dim3 rgrid(std::min((nout + 255) / 256, 64), M);
    splitk_reduce_kernel<<<rgrid, 256, 0, st>>>((float*)workspace, s, M, N, B, Y, ldy, act, g);
    HIP_CHECK_LAUNCH();
    return 0;
  }
  if (f8 && (tsel & 15) >= 5) tsel = (tsel & ~15) | 1;  // 8-wave and mid tiles are bf16-only
  gemm_tiled_plan(M, N, K, &tsel, &s, g != 0);
  static constexpr int kDepth[4] = {2, 3, 4, 6};
  int ns = kDepth[(tsel >> 4) & 3];  // LDS ring depth (hint bits 4-5); bit 6: default-policy weights
  tsel &= 15;
  // the ping-pong kernel's zero-page K tail works on 8-element chunks and its LDS-DMA rows need 16-B aligned
  // strides: anything else runs on the 128x128 tile (tuned hints and C++ callers included, not just linear())
  if (tsel == 4 && (K % 8 || ldx % 8 || ldw % 8)) tsel = 1;
  if ((tsel == 1 || tsel == 5) && ns > 3) ns = 3;  // 128x128 / 256x128 x 4 stages exceed the 160 KiB LDS
  if ((tsel == 2 || tsel == 6) && ns > 4) ns = 4;
  if (f8 && tsel == 4) tsel = 1;
  if (tsel == 4) {
    const bool quad = gemm_quad_ok(N, K, ldx, ldw, 256, Y, ldy, 2, g != 0);
    if (qe && !quad) throw std::runtime_error("gemm: the QKV epilogue of 256 x 256 tiles needs the four-wave kernel");
    if (quad)
      launch_gemm_quad(0, X, ldx, (const bf16_t*)W, ldw, B, Y, ldy, M, N, K, act, g, g_big_group_m,
                       tiles_of(M, N, 256, 256), PpGroup{}, st, qe);
    else
      gemm_pp_kernel<0><<<tiles_of(M, N, 256, 256), 512, 0, st>>>(X, ldx, (const bf16_t*)W, ldw, B, Y, ldy, M, N, K, act, g,
                                                                  g_big_group_m, K & 63 ? zero_page() : nullptr, PpGroup{});
    HIP_CHECK_LAUNCH();
    return 0;
  }
  if ((tsel_raw & 128) && !f8 && tsel < 5) {
    if (launch_streamk(X, ldx, (const bf16_t*)W, ldw, B, Y, ldy, M, N, K, act, g, tsel, ns, s, workspace, ws_bytes,
                       wnt_ok(tsel_raw, M, tsel), st))
      return 0;
    s = 1;  // workspace too small for the partial tiles: plain tiled launch
  }
  int bm, bn;
  tile_dims(tsel, &bm, &bn);
  const int nt = tiles_of(M, N, bm, bn);
  // hint bit 8: split-K slices combine in-launch (last arriver per tile, common.h splitk_combine):
  // slabs [tile][S][bm*bn] in the workspace, finished bf16 output, no reduce launch
  int* cnt = nullptr;
  if ((tsel_raw & 256) && s > 1 && (int64_t)nt * s * bm * bn * 4 <= ws_bytes && Y) cnt = sk_counters(nt);
  if (!cnt && (int64_t)s * M * N * 4 > ws_bytes) s = 1;
  if (qe && (s > 1 && !cnt)) throw std::runtime_error("gemm: the QKV epilogue needs an unsplit or in-launch-combined plan");
  float* part = s > 1 ? (float*)workspace : nullptr;
  const int act_k = s > 1 && !cnt ? 0 : act, glu_k = s > 1 && !cnt ? 0 : g;
  dim3 grid(nt, s);
  if (tsel >= 7 && tsel <= 15) {  // gemm_mid tiles (7, 8-15)
    launch_gemm_mid(tsel, ns, wnt_ok(tsel_raw, M, tsel), X, ldx, (const bf16_t*)W, ldw, B, Y, ldy, part, M, N, K,
                    act_k, glu_k, s, st, cnt, qe, nullptr, nullptr, (tsel_raw & 512) != 0);
    if (cnt) return 0;
    if (s > 1 && partial_out && !g && act == 0) return s;
    if (s > 1) {
      const int nout = g ? N / 2 : N;
      dim3 rgrid(std::min((nout + 255) / 256, 64), M);
      splitk_reduce_kernel<<<rgrid, 256, 0, st>>>(part, s, M, N, B, Y, ldy, act, g);
      HIP_CHECK_LAUNCH();
    }
    return 0;
  }
  // non-temporal weight staging when every weight tile is read by exactly one workgroup row
  const bool wnt = wnt_ok(tsel_raw, M, tsel);
  if (tsel >= 5) {  // 8-wave tiles (bf16 weights)
#define LT8(BM_, BN_, NS_)                                                                                          \
  do {                                                                                                             \
    if (wnt)                                                                                                       \
      gemm_tiled_kernel<BM_, BN_, NS_, true, false, 8><<<grid, 512, 0, st>>>(X, ldx, W, ldw, B, Y, ldy, part, M, N, K, \
                                                                             act_k, glu_k, nullptr, cnt, qv);      \
    else                                                                                                           \
      gemm_tiled_kernel<BM_, BN_, NS_, false, false, 8><<<grid, 512, 0, st>>>(X, ldx, W, ldw, B, Y, ldy, part, M, N,  \
                                                                              K, act_k, glu_k, nullptr, cnt, qv);  \
  } while (0)
    if (tsel == 5) {
      if (ns == 3) LT8(256, 128, 3); else LT8(256, 128, 2);
    } else {
      if (ns == 4) LT8(256, 64, 4); else if (ns == 3) LT8(256, 64, 3); else LT8(256, 64, 2);
    }
#undef LT8
  } else {
#define LT1(BM_, BN_, NS_, WNT_, F8_)                                                                              \
  gemm_tiled_kernel<BM_, BN_, NS_, WNT_, F8_><<<grid, 256, 0, st>>>(X, ldx, W, ldw, B, Y, ldy, part, M, N, K, act_k,  \
                                                                    glu_k, wscale, cnt, qv)
#define LT(BM_, BN_, NS_)                                                                                          \
  do {                                                                                                             \
    if (f8) {                                                                                                      \
      if (wnt) LT1(BM_, BN_, NS_, true, true); else LT1(BM_, BN_, NS_, false, true);                              \
    } else {                                                                                                       \
      if (wnt) LT1(BM_, BN_, NS_, true, false); else LT1(BM_, BN_, NS_, false, false);                            \
    }                                                                                                              \
  } while (0)
  if (ns == 3) {
    if (tsel == 1) LT(128, 128, 3); else if (tsel == 2) LT(64, 128, 3); else LT(64, 64, 3);
  } else if (ns == 4) {
    if (tsel == 2) LT(64, 128, 4); else LT(64, 64, 4);
  } else if (ns == 6) {
    LT(64, 64, 6);
  } else {
    if (tsel == 1) LT(128, 128, 2); else if (tsel == 2) LT(64, 128, 2); else LT(64, 64, 2);
  }
  }
#undef LT
#undef LT1
  HIP_CHECK_LAUNCH();
  if (cnt) return 0;
  if (s > 1 && partial_out && !g && act == 0) return s;
  if (s > 1) {
    const int nout = g ? N / 2 : N;
    dim3 rgrid(std::min((nout + 255) / 256, 64), M);
    splitk_reduce_kernel<<<rgrid, 256, 0, st>>>(part, s, M, N, B, Y, ldy, act, g);
    HIP_CHECK_LAUNCH();
  }
  return 0;
}

// Number of fp32 partial slabs launch_gemm(..., partial_out=true) leaves for these hints, or 0 if
// that call writes the finished output (stream-K, fp8 prefill panels, act / glu epilogues, no
// split). The Python wrapper allocates Y exactly when this returns 0 - one source of truth: the operands are asked for because the plan
// depends on their strides and places (0: strides and places that any plan takes).
int gemm_partial_slabs(int M, int N, int K, bool w_fp8, bool glu, int act, int nt_hint, int split_hint, int64_t ws_bytes,
                       const void* x, int64_t ldx, const void* w, int64_t ldw) {
  if (M == 0 || N == 0 || glu || act != 0) return 0;
  gemm_default_plan(M, N, K, w_fp8, glu, true, ws_bytes, gemm_static_takes(w_fp8, x, ldx, w, ldw), &nt_hint, &split_hint);
  return slabs_of_plan(M, N, K, w_fp8, glu, act, nt_hint, split_hint, ws_bytes);
}

// The same once the hints are those that the launch runs with
static int slabs_of_plan(int M, int N, int K, bool w_fp8, bool glu, int act, int nt_hint, int split_hint, int64_t ws_bytes) {
  if (M == 0 || N == 0 || glu || act != 0) return 0;
  const int tiled_hint = nt_hint >> 8;
  const bool stream = (nt_hint & 0xff) || (!tiled_hint && (M <= 16 || (w_fp8 && M > 128)));
  int s;
  if (stream) {
    if (M > 128) return 0;  // 128-row panels, each finished in place
    int nt;
    gemm_stream_plan(M, N, K, &nt, &s);
    if (split_hint > 0) s = split_hint;
  } else {
    int tsel = tiled_hint;
    if (tsel & kDecHint) {
      if (w_fp8 && !gemm_dec_f8_ok(tsel & 15, M)) return 0;  // rejected at launch
      s = dec_split(M, N, K, split_hint, ws_bytes);
      if (dec_combine_fits(N, tsel, s, ws_bytes)) return 0;  // combined in the launch
      return s > 1 ? s : 0;
    }
    if ((tsel & 128) && !w_fp8 && (tsel & 15) < 5) return 0;  // stream-K combines in-kernel
    if ((tsel & kFourHint) && w_fp8) tsel = split_hint = 0;
    if (tsel & kFourHint) {
      int bm, bn;
      if (!gemm_four_dims(tsel & 15, &bm, &bn)) return 0;  // rejected at launch
      s = std::max(1, split_hint);
      if ((tsel & 256) && (int64_t)tiles_of(M, N, bm, bn) * s * bm * bn * 4 <= ws_bytes) return 0;  // combined in the launch
      return s > 1 && (int64_t)s * M * N * 4 <= ws_bytes ? s : 0;
    }
    if (w_fp8 && ((tsel & 15) == 4 || (tsel & 15) >= 5)) tsel = (tsel & ~15) | 1;
    if ((tsel & 256) && (tsel & 15) != 4) {  // split-K combined in-launch
      int s2 = split_hint, t2 = tsel;
      gemm_tiled_plan(M, N, K, &t2, &s2, false);
      int bm, bn;
      tile_dims(t2 & 15, &bm, &bn);
      if (s2 > 1 && (int64_t)tiles_of(M, N, bm, bn) * s2 * bm * bn * 4 <= ws_bytes) return 0;
    }
    s = split_hint;
    gemm_tiled_plan(M, N, K, &tsel, &s, false);
    if ((tsel & 15) == 4 || (tsel & 128)) return 0;
  }
  if ((int64_t)s * M * N * 4 > ws_bytes) s = 1;
  return s > 1 ? s : 0;
}

// QKV projection with the RoPE + paged-KV write in its LDS-staged epilogue (common.h QkvEpi, tuned kind 3).
// Plan: the hints, else the tuned kind-3 entry, else the static tiled plan; a split plan runs as an in-launch
// combine (the epilogue needs finished sums), a plan of 256 x 256 tiles in the two launches that a product of its size is cut into. Returns -1
// when the shape / plan cannot take the epilogue (stream / stream-K plans, neox RoPE on 256 x 256 tiles or on tiles that are not head-aligned,
// heads that do not divide 256 columns, workspace too small) - the caller then runs the plain GEMM and the rope_cache kernel; 0 when launched.
int launch_gemm_qkv(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, void* y, int64_t ldy,
                    int M, int N, int K, void* workspace, int64_t ws_bytes, int nt_hint, int split_hint,
                    const QkvEpi& qe, hipStream_t st) {
  if (M == 0) return 0;
  if (qe.D <= 0) return -1;
  if (!y) throw std::runtime_error("gemm_qkv: output buffer required");
  if (K % 16) throw std::runtime_error("gemm_qkv: K must be a multiple of 16");
  if (qe.D % 8 || N != (qe.nh + 2 * qe.nkv) * qe.D || N % 8 || ldy % 8) return -1;
  if (qe.do_rope && (qe.rot % 8 || qe.rot > qe.D || (qe.style == 0 && qe.rot % 16))) return -1;
  if (nt_hint == 0 && split_hint == 0) gemm_tuned_get(M, N, K, false, 3, &nt_hint, &split_hint);
  if (nt_hint & 0xff) return -1;  // streaming kernels have no LDS-staged epilogue
  if ((nt_hint >> 8) & kDecHint) {  // decode GEMM: unsplit, or split and combined in the launch (finished sums)
    int bn;
    if (M > 64 || !gemm_dec_bn((nt_hint >> 8) & 15, &bn)) return -1;
    if (qe.do_rope && qe.style == 0 && bn % qe.D) return -1;
    const int s = dec_split(M, N, K, split_hint, ws_bytes);
    const int tsel = (nt_hint >> 8) | (s > 1 ? 256 : 0);
    if (s > 1 && !dec_combine_fits(N, tsel, s, ws_bytes)) return -1;
    launch_tiled((const bf16_t*)x, ldx, w, ldw, (const bf16_t*)bias, (bf16_t*)y, ldy, M, N, K, 0, 0, tsel, s,
                 workspace, ws_bytes, false, st, nullptr, &qe);
    return 0;
  }
  int tsel = nt_hint >> 8, s = split_hint;
  if (tsel & kFourHint) {  // four-wave tiles; a plan that combines split sums in the launch brings no split along (gemm_plan)
    int bm, bn;
    if ((tsel & 256) && s <= 1) {
      const FourPlan p = gemm_four_plan(M, N, K, false, false, ws_bytes);
      tsel = p.hint >> 8, s = p.split;
    }
    if (!gemm_four_ok(N, K, ldx, ldw, y, ldy, false) || !gemm_four_dims(tsel & 15, &bm, &bn) || (s > 1 && !(tsel & 256)) ||
        (qe.do_rope && qe.style == 0 && bn % qe.D))
      return -1;
    if (s > 1 && (int64_t)tiles_of(M, N, bm, bn) * s * bm * bn * 4 > ws_bytes) return -1;
    launch_tiled((const bf16_t*)x, ldx, w, ldw, (const bf16_t*)bias, (bf16_t*)y, ldy, M, N, K, 0, 0, tsel, s, workspace, ws_bytes, false, st,
                 nullptr, &qe);
    return 0;
  }
  gemm_tiled_plan(M, N, K, &tsel, &s, false);
  if (tsel == 4) {  // 256 x 256 tiles, and what they leave over as launch_gemm has it
    if ((qe.do_rope && qe.style != 1) || 256 % qe.D || !gemm_quad_ok(N, K, ldx, ldw, 256, y, ldy, 2, false)) return -1;
    const GemmCut cut = gemm_cut(M, N, K, false, 0);  // unsplit: the epilogue needs finished sums
    const int rows = cut.rows ? cut.rows : M, cols = cut.cols ? cut.cols : N;
    launch_tiled((const bf16_t*)x, ldx, w, ldw, (const bf16_t*)bias, (bf16_t*)y, ldy, rows, cols, K, 0, 0, 4, 1, workspace, ws_bytes, false, st,
                 nullptr, &qe);
    if (rows == M && cols == N) return 0;
    QkvEpi re = qe;  // the rest: its own rows, or the heads from column `cols` on
    if (re.pos) re.pos += rows < M ? rows : 0;
    if (re.slot) re.slot += rows < M ? rows : 0;
    if (cols < N) re.nh -= cols / qe.D;
    const bf16_t* rx = (const bf16_t*)x + (rows < M ? rows * ldx : 0);
    bf16_t* ry = (bf16_t*)y + (rows < M ? rows * ldy : cols);
    const bf16_t* rw = (const bf16_t*)w + (cols < N ? (int64_t)cols * ldw : 0);
    const bf16_t* rb = bias ? (const bf16_t*)bias + (cols < N ? cols : 0) : nullptr;
    const int m = rows < M ? M - rows : M, n = cols < N ? N - cols : N;
    const FourPlan rest = gemm_rest_plan(m, n, K, false, ws_bytes);
    int nt = rest.hint, sp = 1;
    if (!nt) {  // up to 64 rows: the decode kernel where its plan is unsplit, else 64 x 64 tiles
      gemm_static_plan(m, n, K, false, false, ws_bytes, &nt, &sp);
      if (!((nt >> 8) & kDecHint) || sp > 1) nt = 3 << 8;
    }
    launch_tiled(rx, ldx, rw, ldw, rb, ry, ldy, m, n, K, 0, 0, nt >> 8, rest.hint ? rest.split : 1, workspace, ws_bytes, false, st, nullptr, &re);
    return 0;
  }
  if ((tsel & 15) == 4 || (tsel & 128)) return -1;
  int bm, bn;
  tile_dims(tsel & 15, &bm, &bn);
  if (qe.do_rope && qe.style == 0 && bn % qe.D) return -1;  // neox partner columns must share the tile
  if (s > 1) {
    if ((int64_t)tiles_of(M, N, bm, bn) * s * bm * bn * 4 > ws_bytes) return -1;
    tsel |= 256;
  }
  launch_tiled((const bf16_t*)x, ldx, w, ldw, (const bf16_t*)bias, (bf16_t*)y, ldy, M, N, K, 0, 0, tsel, s, workspace,
               ws_bytes, false, st, nullptr, &qe);
  return 0;
}

int launch_gemm_qkv_args(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, void* y, int64_t ldy,
                         int M, int N, int K, void* workspace, int64_t ws_bytes, int nt_hint, int split_hint,
                         const void* pos, const void* cos_t, const void* sin_t, void* kc, void* vc, const void* slot,
                         int nh, int nkv, int D, int rot, int block_size, int style, bool do_rope, hipStream_t st) {
  const QkvEpi qe{(const int64_t*)pos, (const float*)cos_t, (const float*)sin_t, (bf16_t*)kc, (bf16_t*)vc,
                  (const int64_t*)slot, nh, nkv, D, rot, block_size, style, do_rope ? 1 : 0};
  return launch_gemm_qkv(x, ldx, w, ldw, bias, y, ldy, M, N, K, workspace, ws_bytes, nt_hint, split_hint, qe, st);
}

void gemm_plan(int M, int N, int K, bool w_fp8, bool glu, bool slabs, int* nt, int* splitk, bool four);
void gemm_cut_of(int M, int N, int K, bool glu, int* rows, int* cols, int* split) {
  const GemmCut c = gemm_cut(M, N, K, glu, 64 << 20);
  *rows = c.rows;
  *cols = c.cols;
  *split = c.rows || c.cols ? std::max(1, gemm_rest_plan(c.rows ? M - c.rows : M, c.cols ? N - c.cols : N, K, glu, 64 << 20).split) : 1;
}

// The plan of a product whose result goes straight into an op that can sum its slabs: a split one, the slabs unsummed, where the older rules
// split K of the finished product, so that it stays in 32 bits there; else split 1, and the product is finished by the plan of its size. A tuned
// plan stays as it is. The four-wave tiles' slabs against the older tiles', with the closing op: 0.90 of the time over 582 products of 17 - 64 rows,
// 1.02 at worst, and where the older tiles had those of 17 - 32 rows and K beyond 5120 to themselves 0.83 over 229, none slower (us, 21 x 2048 x 5632
// 12.9 and 12.2, 28 x 2048 x 11264 17.6 and 16.9).
void gemm_closing_plan(int M, int N, int K, int* nt, int* splitk) {
  int tuned_nt, tuned_split;
  gemm_plan(M, N, K, false, false, false, nt, splitk, false);
  if (gemm_tuned_get(M, N, K, false, 0, &tuned_nt, &tuned_split)) return;
  if (*splitk <= 1) return;
  const FourPlan p = gemm_four_plan(M, N, K, false, true, 64 << 20);
  if (p.hint) *nt = p.hint, *splitk = p.split;
}

// The plan of a product without hints. slabs: of one whose consumer sums split-K slabs itself
void gemm_plan(int M, int N, int K, bool w_fp8, bool glu, bool slabs, int* nt, int* splitk, bool four) {
  *nt = *splitk = 0;
  const bool tuned = gemm_tuned_get(M, N, K, glu, w_fp8 ? 1 : 0, nt, splitk);
  if (!tuned && w_fp8) gemm_static_plan_f8(M, N, K, glu, slabs && !glu, 64 << 20, nt, splitk);
  else if (!tuned) gemm_static_plan(M, N, K, glu, slabs && !glu, 64 << 20, nt, splitk, four);
  if (tuned || *nt) {
    if ((*nt >> 8) & kDecHint) {
      *splitk = ((*nt >> 8) & 256) ? 1 : dec_split(M, N, K, *splitk, INT64_MAX);
    } else if ((*nt >> 8) & (128 | 256)) {
      *splitk = 1;  // stream-K / split-K combine finish their tiles in-kernel: no partial slabs for the consumer
    } else if ((*nt >> 8) && !((*nt >> 8) & kFourHint)) {  // tiled hint: the split the kernel will really use
      int tsel = *nt >> 8;
      gemm_tiled_plan(M, N, K, &tsel, splitk, glu);
    }
    return;
  }
  if (M <= 16 || (w_fp8 && M > 128)) {
    gemm_stream_plan(std::min(M, 128), N, K, nt, splitk);
  } else {
    int tsel = 0, s = 0;
    gemm_tiled_plan(M, N, K, &tsel, &s, glu);
    *nt = tsel << 8;
    *splitk = s;
  }
}

// Whether grouped products of launch_moe_pp's modes take the four-wave kernel
bool moe_pp_quad(int mode, int64_t lda, int maxt, int top, int N, int K, const void* C) {
  return gemm_quad_ok(N, K, lda, K, mode == 2 ? 256 : (int64_t)maxt * 256 / std::max(top, 1) + 1, C, mode == 3 ? N / 2 : N, mode == 2 ? 4 : 2,
                      mode == 3, true);
}

// Grouped expert products on 256 x 256 tiles (gemm_quad.hip, else the ping-pong kernel), over a tile list of 256 rows per tile whose taller tiles
// stand first, their number behind it (launch_moe_group with `tall`): C = act(A[order / top] W_e^T) in bf16 (mode 1), C = A W_e^T in fp32 (mode
// 2), or C [rows, N / 2] = silu(gate) * up in bf16 with W's rows gate and up in alternating groups of 16 (mode 3). A [rows, K] with row stride
// lda, W [E, N, K].
void launch_moe_pp(int mode, const void* A, int64_t lda, const void* W, const void* meta, const void* order, void* C, int E,
                   int maxt, int top, int N, int K, int act, hipStream_t st) {
  if (maxt <= 0) return;
  if (K % 8 || lda % 8 || (((uintptr_t)A | (uintptr_t)W) & 15)) throw std::runtime_error("moe_pp: rows must be 16-byte aligned");
  const int64_t nwg = (int64_t)maxt * ((N + 255) / 256);
  if (nwg > 0x7fffffff) throw std::runtime_error("moe_pp: grid too large");
  PpGroup gr;
  gr.meta = (const int*)meta, gr.order = (const int*)order, gr.E = E, gr.maxt = maxt, gr.top = top;
  gr.sB = (int64_t)N * K;
  gr.Yf = (float*)C;
  const char* z = K & 63 ? zero_page() : nullptr;
  const int glu = mode == 3;
  if (glu && N % 32) throw std::runtime_error("moe_pp: gate and up in groups of 16 rows");
  if (moe_pp_quad(mode, lda, maxt, top, N, K, C)) {
    if (mode < 1 || mode > 3) throw std::runtime_error("moe_pp: mode");
    launch_gemm_quad(mode == 2 ? 2 : 1, (const bf16_t*)A, lda, (const bf16_t*)W, K, nullptr, (bf16_t*)C, glu ? N / 2 : N, 0, N, K,
                     glu ? 0 : act, glu, 1, (unsigned)nwg, gr, st);
    return;
  }
#define LAUNCH_PPG(G_)                                                                                              \
  gemm_pp_kernel<G_><<<(unsigned)nwg, 512, 0, st>>>((const bf16_t*)A, lda, (const bf16_t*)W, K, nullptr, (bf16_t*)C, \
                                                    glu ? N / 2 : N, 0, N, K, glu ? 0 : act, glu, 1, z, gr)
  if (mode == 1 || mode == 3) LAUNCH_PPG(1);
  else if (mode == 2) LAUNCH_PPG(2);
  else throw std::runtime_error("moe_pp: mode");
#undef LAUNCH_PPG
  HIP_CHECK_LAUNCH();
}

// Whether moe_pp_glu takes a layer with gate and up matrices [E, F, K] of their own: h [rows, K] with row stride ldh.
bool moe_pp_glu_ok(int64_t ldh, int maxt, int top, int F, int K) {
  return gemm_quad_ok(2 * F, K, ldh, K, (int64_t)maxt * 256 / std::max(top, 1) + 1, nullptr, F, 2, true, true) && F % 16 == 0;
}

// act [pairs, F] = glu(pw h Wg_e^T, pw h Wu_e^T) in bf16 over launch_moe_pp's tile list
void launch_moe_pp_glu(const void* h, int64_t ldh, const void* Wg, const void* Wu, const void* meta, const void* order, void* act,
                       int E, int maxt, int top, int F, int K, float limit, float alpha, const void* pw, int silu, hipStream_t st) {
  if (maxt <= 0) return;
  if (!moe_pp_glu_ok(ldh, maxt, top, F, K) || (((uintptr_t)h | (uintptr_t)Wg | (uintptr_t)Wu | (uintptr_t)act) & 15))
    throw std::runtime_error("moe_pp_glu: K % 64, F % 16, rows of 16-byte alignment");
  const int64_t nwg = (int64_t)maxt * ((2 * F + 255) / 256);
  if (nwg > 0x7fffffff) throw std::runtime_error("moe_pp_glu: grid too large");
  PpGroup gr;
  gr.meta = (const int*)meta, gr.order = (const int*)order, gr.E = E, gr.maxt = maxt, gr.top = top;
  gr.sB = (int64_t)F * K;
  gr.Wu = (const bf16_t*)Wu, gr.pw = (const float*)pw, gr.limit = limit, gr.alpha = alpha, gr.silu = silu;
  launch_gemm_quad(3, (const bf16_t*)h, ldh, (const bf16_t*)Wg, K, nullptr, (bf16_t*)act, F, 0, 2 * F, K, 0, 1, 1, (unsigned)nwg, gr,
                   st);
}
