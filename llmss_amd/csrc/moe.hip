// Mixture-of-experts feed-forward: routing, grouping of (token, expert) pairs and the grouped expert GEMMs.
//
//   z = W_router h (fp32, gemm_any)                                   [T, E]
//   moe_route:   s = sigmoid(z), or softmax(z) over all experts; the `top` experts with the largest s + correction are chosen (ties: the lower
//                index); weights = chosen s / (their sum + 1e-20)     -> idx [T, top] int32, wts [T, top] fp32
//                or (score 2) s = z, the chosen ones weighted by a softmax over themselves. A bias may be added to z; one
//                more column of z after the E routed ones may hold a gate, whose sigmoid goes to sg [T]
//                A router may have more outputs than there are experts: the outputs from E on are identity experts,
//                whose output is the layer's input row; their pairs are left out of the grouping (place -1).
//   moe_group:   pairs p = t * top + j are bucketed by expert: off [E + 1], order [P] (pair at each sorted row),
//                place [P] (sorted row of each pair) and a flat list of row tiles (expert, first row; 64 or 128 rows each) so the
//                grouped GEMMs launch a grid whose size is known on the host (ceil(P / rows) + E tiles at most)
//   moe_gate_up: act[r, f] = glu(h[token(r)] . gate_e[f], h[token(r)] . up_e[f])   for sorted row r of expert e
//   moe_down:    y[r, n] = act[r, :] . down_e[n, :]                   (fp32)
//   moe_combine: out[t, :] = sum_j wts[t, j] * y[place[t * top + j], :] (+ (sw[t] *) shared[t, :])   (fp32, j ascending;
//                no wts: the plain sum, for layers whose weights went onto the experts' inputs in moe_gate_up)
//
// Expert activation (clamped, gated): g = min(g, limit), u = clamp(u, -limit, limit),
// glu = g * sigmoid(alpha * g) * (u + 1). glu_clamp applies the same to a dense [T, 2F] gate|up product (the
// shared expert, which runs through the ordinary GEMMs).
//
// Nothing here synchronises with the host: group sizes stay on the device, so a decode step with experts can be
// captured into a HIP graph. Every pair's row is computed alone, so a token's result does not depend on what else
// is in the step.
#include "anytype.h"
#include "route.h"
#include "tile_valu.h"

__device__ __forceinline__ float glu_clamped(float g, float u, float limit, float alpha) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + 1.f);
}
// silu: the plain gated form silu(g) * u, no clamps
__device__ __forceinline__ float glu_value(float g, float u, float limit, float alpha, int silu) {
  return silu ? g / (1.f + expf(-g)) * u : glu_clamped(g, u, limit, alpha);
}

// ------------------------------------------------------------------------------------------------ routing
// one wave per token; lanes over experts
__global__ __launch_bounds__(64) void moe_route_kernel(const float* __restrict__ z, const float* __restrict__ corr,
                                                       int* __restrict__ idx, float* __restrict__ wts, int E, int top,
                                                       int norm, int smax, const float* __restrict__ zb,
                                                       float* __restrict__ sg) {
  extern __shared__ __attribute__((aligned(16))) float sc[];  // [E] scores, [E] choice values
  float* ch = sc + E;
  const int t = blockIdx.x, lane = threadIdx.x;
  const float* zr = z + (int64_t)t * (E + (sg ? 1 : 0));
  if (sg && lane == 0) sg[t] = 1.f / (1.f + expf(-zr[E]));
  if (E <= 128) {
    float v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) v[j] = lane + 64 * j < E ? zr[lane + 64 * j] + (zb ? zb[lane + 64 * j] : 0.f) : -INFINITY;
    route_ranked(v, sc, corr, idx + (int64_t)t * top, wts + (int64_t)t * top, E, top, norm, smax);
    return;
  }
  float mx = 0.f, den = 1.f;
  if (smax == 1) {
    mx = -INFINITY, den = 0.f;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, zr[e] + (zb ? zb[e] : 0.f));
    mx = warp_max(mx);
    for (int e = lane; e < E; e += 64) den += expf(zr[e] + (zb ? zb[e] : 0.f) - mx);
    den = warp_sum(den);
  }
  for (int e = lane; e < E; e += 64) {
    const float ze = zr[e] + (zb ? zb[e] : 0.f);
    const float s = smax == 2 ? ze : smax ? expf(ze - mx) / den : 1.f / (1.f + expf(-ze));
    sc[e] = s;
    ch[e] = s + (corr ? corr[e] : 0.f);
  }
  __syncthreads();
  float sum = 0.f, first = 0.f;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float v = ch[e];
      if (v > best || (v == best && e < bi)) {
        best = v;
        bi = e;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > best || (ov == best && oi < bi)) {
        best = ov;
        bi = oi;
      }
    }
    if (bi >= E) bi = 0;  // every value NaN: keep indices in range
    float s = sc[bi];
    if (smax == 2) {  // the first one chosen is the largest
      if (j == 0) first = s;
      s = expf(s - first);
    }
    sum += s;
    if (lane == 0) {
      idx[(int64_t)t * top + j] = bi;
      wts[(int64_t)t * top + j] = s;
      ch[bi] = -INFINITY;
    }
    __syncthreads();
  }
  if (!norm && smax != 2) return;  // the chosen scores themselves
  const float inv = 1.f / (sum + (smax == 2 ? 0.f : 1e-20f));
  for (int j = lane; j < top; j += 64) wts[(int64_t)t * top + j] *= inv;
}

void launch_moe_route(const void* z, const void* corr, void* idx, void* wts, int T_, int E, int top, int norm,
                      int smax, const void* zb, void* sg, hipStream_t st) {
  if (T_ == 0) return;
  if (top > E || top <= 0) throw std::runtime_error("moe_route: top must be in [1, experts]");
  moe_route_kernel<<<T_, 64, (2 * E + 4) * sizeof(float), st>>>((const float*)z, (const float*)corr, (int*)idx, (float*)wts,
                                                           E, top, norm, smax, (const float*)zb, (float*)sg);
  HIP_CHECK_LAUNCH();
}

// Router logits and routing in one launch, for steps of few tokens (a decode step): one workgroup per token, its waves
// share the experts' dot products z_e = h . W_r[e] (fp32 accumulation over lanes), then the token is routed
// as moe_route_kernel does. A prompt's thousands of tokens take the matrix-core GEMM and moe_route instead.
// Bound by the chain of a wave's reads (the weights are cold: the layer's experts went through the caches since), so the row and up to
// three outputs' weights are asked for at once. 33 rows of
// 2048, 33 outputs: 10.2 -> 6.6 us, 8 rows of 1024, 17 outputs: 5.1 -> 3.9 (each with the faster routing above)
template <typename T>
__global__ __launch_bounds__(1024) void moe_router_kernel(const T* __restrict__ h, int64_t ldh, const T* __restrict__ wr,
                                                         const float* __restrict__ corr, int* __restrict__ idx,
                                                         float* __restrict__ wts, int E, int K, int top, bool vec,
                                                         int norm, int smax, const float* __restrict__ zb,
                                                         float* __restrict__ sg) {
  extern __shared__ __attribute__((aligned(16))) float sc[];  // [E] scores, [E] choice values
  float* ch = sc + E;
  const bool ranked = E <= 128;
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
  const T* x = h + (int64_t)t * ldh;
  const int EG = E + (sg ? 1 : 0);
  auto put = [&](int e, float acc) {  // (one lane) an output's sum over K
    if (e == E) {
      sg[t] = 1.f / (1.f + expf(-acc));
      return;
    }
    if (zb) acc += zb[e];
    if (ranked) {
      sc[e] = acc;
      return;
    }
    const float s = smax ? acc : 1.f / (1.f + expf(-acc));
    sc[e] = s;
    ch[e] = s + (corr ? corr[e] : 0.f);
  };
  if (vec) {  // K % 8 == 0, rows 16-byte aligned - eight elements per lane, two or four 16-byte accesses
    typedef T vec8 __attribute__((ext_vector_type(8)));
    constexpr int U = sizeof(T) == 2 ? 4 : 2;  // chunks of 512 numbers in flight
    auto dots = [&](int e0, auto n_c) {        // outputs e0, e0 + nw, ..
      constexpr int NE = decltype(n_c)::value;
      float acc[NE];
#pragma unroll
      for (int n = 0; n < NE; ++n) acc[n] = 0.f;
      for (int k0 = lane * 8; k0 < K; k0 += 512 * U) {
        vec8 xv[U], wt[NE][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = min(k0 + 512 * u, K - 8);
          xv[u] = *reinterpret_cast<const vec8*>(x + k);
#pragma unroll
          for (int n = 0; n < NE; ++n) wt[n][u] = *reinterpret_cast<const vec8*>(wr + (int64_t)(e0 + n * nw) * K + k);
        }
        __builtin_amdgcn_sched_barrier(0);  // all loads are issued before the first sum waits for one
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (k0 + 512 * u >= K) break;
#pragma unroll
          for (int n = 0; n < NE; ++n)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const T xi = xv[u][i], wi = wt[n][u][i];
              acc[n] = fmaf(El<T>::ld(&xi), El<T>::ld(&wi), acc[n]);
            }
        }
      }
#pragma unroll
      for (int n = 0; n < NE; ++n) {
        acc[n] = warp_sum(acc[n]);
        if (lane == 0) put(e0 + n * nw, acc[n]);
      }
    };
    for (int e0 = wv; e0 < EG; e0 += 3 * nw) {
      if (e0 + 2 * nw < EG) dots(e0, std::integral_constant<int, 3>{});
      else if (e0 + nw < EG) dots(e0, std::integral_constant<int, 2>{});
      else dots(e0, std::integral_constant<int, 1>{});
    }
  } else {
    for (int e = wv; e < EG; e += nw) {
      const T* w = wr + (int64_t)e * K;
      float acc = 0.f;
      for (int k = lane; k < K; k += 64) acc = fmaf(El<T>::ld(x + k), El<T>::ld(w + k), acc);
      acc = warp_sum(acc);
      if (lane == 0) put(e, acc);
    }
  }
  __syncthreads();
  if (ranked) {
    if (wv) return;
    float v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) v[j] = lane + 64 * j < E ? sc[lane + 64 * j] : -INFINITY;
    __builtin_amdgcn_wave_barrier();
    route_ranked(v, sc, corr, idx + (int64_t)t * top, wts + (int64_t)t * top, E, top, norm, smax);
    return;
  }
  if (smax == 1) {  // sc holds the logits: every wave forms their maximum and sum, then the scores replace them
    float mx = -INFINITY, den = 0.f;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, sc[e]);
    mx = warp_max(mx);
    for (int e = lane; e < E; e += 64) den += expf(sc[e] - mx);
    den = warp_sum(den);
    __syncthreads();
    for (int e = tid; e < E; e += blockDim.x) {
      const float s = expf(sc[e] - mx) / den;
      sc[e] = s;
      ch[e] = s + (corr ? corr[e] : 0.f);
    }
    __syncthreads();
  }
  float sum = 0.f, first = 0.f;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float v = ch[e];
      if (v > best || (v == best && e < bi)) {
        best = v;
        bi = e;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > best || (ov == best && oi < bi)) {
        best = ov;
        bi = oi;
      }
    }
    if (bi >= E) bi = 0;
    float s = sc[bi];
    if (smax == 2) {
      if (j == 0) first = s;
      s = expf(s - first);
    }
    sum += s;
    __syncthreads();  // every wave has read ch before the winner is struck out
    if (tid == 0) {
      idx[(int64_t)t * top + j] = bi;
      wts[(int64_t)t * top + j] = s;
      ch[bi] = -INFINITY;
    }
    __syncthreads();
  }
  if (!norm && smax != 2) return;
  const float inv = 1.f / (sum + (smax == 2 ? 0.f : 1e-20f));
  for (int j = tid; j < top; j += blockDim.x) wts[(int64_t)t * top + j] *= inv;
}

void launch_moe_router(const void* h, int64_t ldh, const void* wr, const void* corr, void* idx, void* wts, int T_,
                       int E, int K, int top, int dt, int norm, int smax, const void* zb, void* sg, hipStream_t st) {
  if (T_ == 0) return;
  if (top > E || top <= 0) throw std::runtime_error("moe_router: top must be in [1, experts]");
  const int es = dt == 0 ? 2 : 4;
  const bool vec = K % 8 == 0 && ((uintptr_t)h % 16) == 0 && ((uintptr_t)wr % 16) == 0 && (ldh * es) % 16 == 0;
  const int threads = E >= 16 ? 1024 : (E >= 8 ? 512 : 256);  // a wave per expert up to 16 waves
  DISPATCH_T(dt, T, (moe_router_kernel<T><<<T_, threads, (2 * E + 4) * sizeof(float), st>>>(
                        (const T*)h, ldh, (const T*)wr, (const float*)corr, (int*)idx, (float*)wts, E, K, top, vec,
                        norm, smax, (const float*)zb, (float*)sg)));
  HIP_CHECK_LAUNCH();
}

// The same for bf16 rows on the matrix cores, at any number of rows: a workgroup takes 16 tokens and all outputs (up to 16 *
// MR_NT), its eight waves an eighth of K each (fragments straight from memory: lane (li, g) holds k = 8 g .. 8 g + 7 of row li);
// the parts meet in LDS and every wave routes two of the tokens, a score per lane (lane e: outputs e, e + 64) whose rank among
// all decides whether and where it is chosen.
#define MR_NT 8
template <int NT>
__global__ __launch_bounds__(512) void moe_router_mfma_kernel(const bf16_t* __restrict__ h, int64_t ldh,
                                                              const bf16_t* __restrict__ wr, const float* __restrict__ corr,
                                                              int* __restrict__ idx, float* __restrict__ wts, int T_, int E,
                                                              int K, int top, int norm, int smax,
                                                              const float* __restrict__ zb, float* __restrict__ sg) {
  constexpr int LD = 16 * NT + 4;
  __shared__ __attribute__((aligned(16))) float part[4][16][LD];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16, EG = E + (sg ? 1 : 0);
  f32x4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16_t* a = h + (int64_t)min(t0 + li, T_ - 1) * ldh + 8 * g;
  const bf16_t* b[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) b[j] = wr + (int64_t)min(16 * j + li, EG - 1) * K + 8 * g;
  const int ks = K / 32;  // (neighbouring waves take neighbouring steps: the halves of a 128-byte line meet in the cache)
  constexpr int U = NT <= 4 ? 8 : 4;  // steps whose loads are in flight together
  for (int k0 = w; k0 < ks; k0 += 8 * U) {  // (K a multiple of 32; steps past the end repeat the last one with a zero row)
    s16x8 av[U], bv[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + 8 * u, ks - 1);
      av[u] = *reinterpret_cast<const s16x8*>(a + 32 * k);
#pragma unroll
      for (int j = 0; j < NT; ++j) bv[u][j] = *reinterpret_cast<const s16x8*>(b[j] + 32 * k);
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads are issued before the first product waits for one
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + 8 * u >= ks) av[u] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u], bv[u][j], acc[j], 0, 0, 0);
    }
  }
  if (w >= 4) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[w - 4][4 * g + i][16 * j + li] = acc[j][i];
  }
  __syncthreads();
  if (w < 4) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[w][4 * g + i][16 * j + li] += acc[j][i];
  }
  __syncthreads();
  auto z_of = [&](int r, int e) { return (part[0][r][e] + part[1][r][e]) + (part[2][r][e] + part[3][r][e]); };
  for (int r = 2 * w; r < 2 * w + 2; ++r) {
    const int64_t t = t0 + r;
    if (t >= T_) return;
    float sc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = lane + 64 * j;
      sc[j] = e < E ? z_of(r, e) + (zb ? zb[e] : 0.f) : -INFINITY;
    }
    if (sg && lane == 0) sg[t] = 1.f / (1.f + expf(-z_of(r, E)));
    __builtin_amdgcn_wave_barrier();
    route_ranked(sc, &part[0][r][0], corr, idx + t * top, wts + t * top, E, top, norm, smax);  // (the row is this wave's alone)
  }
}

// Up to 48 outputs: both operands through LDS. The form above reads 16 bytes of 16 rows side by side, neighbouring lanes in different
// rows, and gets 12 KB a microsecond into a CU; here a wave reads whole kilobytes of a row, 512 numbers of 16 * TG tokens and all outputs
// a stage (rows dealt to the waves), the next stage in registers behind the products of this one. A wave's products are two of a stage's
// sixteen steps of 32; parts and routing as above. Rows of 520 numbers in LDS: 16 rows' pieces lie in 64 different banks. 8261 rows of
// 2048, 33 outputs: 41.6 -> 15.5 us, 8192 rows, 32 outputs: 20.6 -> 11.4, 300 rows: 15.0 -> 7.5.
template <int OR, int TG>
__global__ __launch_bounds__(512, 4) void moe_router_tile_kernel(const bf16_t* __restrict__ h, int64_t ldh,
                                                                 const bf16_t* __restrict__ wr, const float* __restrict__ corr,
                                                                 int* __restrict__ idx, float* __restrict__ wts, int T_, int E,
                                                                 int K, int top, int norm, int smax,
                                                                 const float* __restrict__ zb, float* __restrict__ sg) {
  constexpr int NT = (OR + 15) / 16, LD = 16 * NT + 4, KS = 512, LDK = KS + 8, ROWS = 16 * TG + OR, NL = ROWS / 8;
  constexpr int BYTES = ROWS * LDK * 2 > 4 * 16 * TG * LD * 4 ? ROWS * LDK * 2 : 4 * 16 * TG * LD * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[BYTES];
  bf16_t* st = reinterpret_cast<bf16_t*>(smem);                    // [ROWS][LDK]: tokens, then outputs
  float(*part)[16 * TG][LD] = reinterpret_cast<float(*)[16 * TG][LD]>(smem);  // (after the last product)
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16 * TG, EG = E + (sg ? 1 : 0);
  f32x4 acc[TG][NT];
#pragma unroll
  for (int n = 0; n < TG; ++n)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[n][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u16x8 v[NL];
  auto load = [&](int k0) {
    const int k = min(k0 + lane * 8, K - 8);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int r = w + 8 * i;  // (16 * TG is a multiple of 8: a load is of tokens or of outputs in every wave)
      const bf16_t* row = i < 2 * TG ? h + (int64_t)min(t0 + r, T_ - 1) * ldh : wr + (int64_t)min(r - 16 * TG, EG - 1) * K;
      v[i] = *reinterpret_cast<const u16x8*>(row + k);
    }
  };
  load(0);
  for (int k0 = 0; k0 < K; k0 += KS) {
    if (k0) __syncthreads();  // every wave has read the stage before
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<u16x8*>(st + (w + 8 * i) * LDK + lane * 8) = v[i];
    __syncthreads();
    if (k0 + KS < K) load(k0 + KS);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int ks = w + 8 * u;
      if (k0 + 32 * ks >= K) break;  // (K a multiple of 32)
      s16x8 av[TG], bv[NT];
#pragma unroll
      for (int n = 0; n < TG; ++n) av[n] = *reinterpret_cast<const s16x8*>(st + (16 * n + li) * LDK + 32 * ks + 8 * g);
#pragma unroll
      for (int j = 0; j < NT; ++j) bv[j] = *reinterpret_cast<const s16x8*>(st + min(16 * (TG + j) + li, ROWS - 1) * LDK + 32 * ks + 8 * g);
#pragma unroll
      for (int n = 0; n < TG; ++n)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[n][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[n], bv[j], acc[n][j], 0, 0, 0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int half = 0; half < 2; ++half) {  // waves 4 - 7 leave theirs, then 0 - 3 add their own
    if (half ? w < 4 : w >= 4) {
#pragma unroll
      for (int n = 0; n < TG; ++n)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float& z = part[w & 3][16 * n + 4 * g + i][16 * j + li];
            z = half ? z + acc[n][j][i] : acc[n][j][i];
          }
    }
    __syncthreads();
  }
  // a wave routes 2 * TG tokens, as many at once as groups of lanes fit (the gate's output is one of the columns, none of the experts)
  auto route = [&](auto lanes_c) {
    constexpr int LN = decltype(lanes_c)::value;
    const int e = lane & (LN - 1);
    float cr[1] = {corr && e < E ? corr[e] : 0.f};
    const float b = zb && e < E ? zb[e] : 0.f;
#pragma unroll
    for (int r0 = 0; r0 < 2 * TG; r0 += 64 / LN) {
      const int r = 2 * TG * w + r0 + lane / LN;
      const int64_t t = t0 + r;
      if (r0 + lane / LN >= 2 * TG || t >= T_) continue;
      auto z_of = [&](int c) { return (part[0][r][c] + part[1][r][c]) + (part[2][r][c] + part[3][r][c]); };
      float sc[1] = {e < E ? z_of(e) + b : -INFINITY};
      if (sg && e == 0) sg[t] = 1.f / (1.f + expf(-z_of(E)));
      __builtin_amdgcn_wave_barrier();
      route_ranked<LN, 1>(sc, cr, &part[0][r][0], idx + t * top, wts + t * top, E, top, norm, smax);  // (the row is this group's alone)
    }
  };
  if (E <= 16) route(std::integral_constant<int, 16>{});
  else if (E <= 32) route(std::integral_constant<int, 32>{});
  else route(std::integral_constant<int, 64>{});
}

// may a router of E outputs (+ gate) over bf16 rows of K numbers take the matrix-core form?
bool moe_router_mfma_ok(int E, int gate, int K) { return E + (gate ? 1 : 0) <= 16 * MR_NT && E <= 128 && K % 32 == 0; }

void launch_moe_router_mfma(const void* h, int64_t ldh, const void* wr, const void* corr, void* idx, void* wts, int T_,
                            int E, int K, int top, int norm, int smax, const void* zb, void* sg, hipStream_t st) {
  if (T_ == 0) return;
  if (top > E || top <= 0) throw std::runtime_error("moe_router: top must be in [1, experts]");
  if (!moe_router_mfma_ok(E, sg != nullptr, K) || (((uintptr_t)h | (uintptr_t)wr) & 15) || ldh % 8)
    throw std::runtime_error("moe_router: shape of the matrix-core form");
#define LAUNCH_MR(NT_)                                                                                                      \
  moe_router_mfma_kernel<NT_><<<(T_ + 15) / 16, 512, 0, st>>>((const bf16_t*)h, ldh, (const bf16_t*)wr, (const float*)corr, \
                                                              (int*)idx, (float*)wts, T_, E, K, top, norm, smax,            \
                                                              (const float*)zb, (float*)sg)
#define LAUNCH_MRT(OR_, TG_)                                                                                              \
  moe_router_tile_kernel<OR_, TG_><<<(T_ + 16 * TG_ - 1) / (16 * TG_), 512, 0, st>>>(                                     \
      (const bf16_t*)h, ldh, (const bf16_t*)wr, (const float*)corr, (int*)idx, (float*)wts, T_, E, K, top, norm, smax,    \
      (const float*)zb, (float*)sg)
#define LAUNCH_MRT_T(OR_)              \
  do {                                 \
    if (two) LAUNCH_MRT(OR_, 2);       \
    else LAUNCH_MRT(OR_, 1);           \
  } while (0)
  const int eg = E + (sg ? 1 : 0);
  const bool two = T_ > 4096;  // (until then 16 tokens a workgroup are a CU's share: 4096 rows of 2048 8.8 us, 4097 rows 11.1)
  if (eg <= 16) LAUNCH_MRT_T(16);
  else if (eg <= 32) LAUNCH_MRT_T(32);
  else if (eg <= 40) LAUNCH_MRT_T(40);  // (two workgroups of 32 tokens to a CU's LDS)
  else if (eg <= 48) LAUNCH_MRT_T(48);
  else if (eg <= 80) LAUNCH_MR(5);
  else LAUNCH_MR(MR_NT);
#undef LAUNCH_MRT_T
#undef LAUNCH_MRT
#undef LAUNCH_MR
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ grouping
// meta = [ntiles | off[E + 1] | tile_expert[maxt] | tile_row0[maxt]], order [P], place [P].
// One wave turns the experts' counts into their first rows (off, and `cur` in LDS for the caller's own use) and the list of tiles: a lane an
// expert, sums over the lanes. meta null: only `cur`. tall: the list in two parts, first the tiles of more than half of their rows, whose number
// lies behind the list, then the others (gemm_quad.hip).
__device__ __forceinline__ void group_scan(const int* cnt, int* cur, int E, int maxt, int tile_rows, int* meta, int tall) {
  const int lane = threadIdx.x & 63;
  int* off = meta + 1;
  int* tile_e = meta + 1 + (E + 1);
  int* tile_r = tile_e + maxt;
  int o = 0, nt = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane, c = e < E ? cnt[e] : 0, t = (c + (tall ? tile_rows - tile_rows / 2 : tile_rows) - 1) / tile_rows;
    int so = c, st = t;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int uo = __shfl_up(so, d, 64), ut = __shfl_up(st, d, 64);
      so += lane >= d ? uo : 0;
      st += lane >= d ? ut : 0;
    }
    const int eo = o + so - c, et = nt + st - t;
    if (e < E) {
      cur[e] = eo;
      if (meta) {
        off[e] = eo;
        for (int i = 0; i < t && et + i < maxt; ++i) {
          tile_e[et + i] = e;
          tile_r[et + i] = eo + i * tile_rows;
        }
      }
    }
    o += __shfl(so, 63, 64);
    nt += __shfl(st, 63, 64);
  }
  if (tall && meta) {
    if (lane == 0) meta[2 + E + 2 * (int64_t)maxt] = nt < maxt ? nt : maxt;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane, c = e < E ? cnt[e] : 0, rest = c % tile_rows;
      const uint64_t some = __ballot(rest > 0 && 2 * rest <= tile_rows);
      const int at = nt + __popcll(some & ((1ull << lane) - 1));
      if ((some >> lane & 1) && at < maxt) {
        tile_e[at] = e;
        tile_r[at] = off[e] + c - rest;
      }
      nt += __popcll(some);
    }
  }
  if (meta && lane == 0) {
    off[E] = o;
    meta[0] = nt < maxt ? nt : maxt;
  }
}

// One workgroup, for steps of few pairs. Bound by its chain: the counts, their sums, the rows. (With the sums formed by one thread, an
// expert after the other, and the pairs read twice: 132 pairs of 32 experts 6.3 us, 2.7 here.)
__global__ __launch_bounds__(1024) void moe_group_kernel(const int* __restrict__ idx, int P, int E, int maxt,
                                                         int* __restrict__ meta, int* __restrict__ order,
                                                         int* __restrict__ place, int tile_rows, int tall) {
  extern __shared__ int sm[];  // cnt[E], cur[E]
  int* cnt = sm;
  int* cur = sm + E;
  for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  constexpr int U = 8;  // pairs per thread whose loads and atomics are in flight together
  int e[U];
  for (int p0 = threadIdx.x; p0 < P; p0 += blockDim.x * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * blockDim.x;
      e[u] = p < P ? idx[p] : E;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e[u] < E) atomicAdd(&cnt[e[u]], 1);
  }
  __syncthreads();
  if (threadIdx.x < 64) group_scan(cnt, cur, E, maxt, tile_rows, meta, tall);
  __syncthreads();
  // rows within an expert take whatever order the atomics give: every pair's row is computed on its own, so the
  // values do not depend on where the row lands
  const bool again = P > (int)blockDim.x * U;  // (else the experts are still at hand)
  for (int p0 = threadIdx.x; p0 < P; p0 += blockDim.x * U) {
    int o[U];
    if (again) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int p = p0 + u * blockDim.x;
        e[u] = p < P ? idx[p] : E;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) o[u] = e[u] < E ? atomicAdd(&cur[e[u]], 1) : -1;  // (-1: an identity expert, no row of its own)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * blockDim.x;
      if (p >= P) continue;
      if (o[u] >= 0) order[o[u]] = p;
      place[p] = o[u];
    }
  }
}

// Many pairs: 1024 of them a workgroup. One launch leaves every workgroup's counts behind `meta`, the next sums those of all workgroups and
// of the ones before its own, and hands out the rows from there. One workgroup alone is bound by its LDS atomics, two a pair:
// 33044 pairs of 32 experts 46 us with the sums above by one thread, 19.6, in two launches 6.0; 2048 pairs 3.4 and 4.4, 4096 pairs 4.4
// and 4.8, 8192 pairs 6.5 and 5.1.
__global__ __launch_bounds__(1024) void moe_count_kernel(const int* __restrict__ idx, int P, int E, int* __restrict__ hist) {
  extern __shared__ int sm[];  // cnt[E]
  for (int e = threadIdx.x; e < E; e += 1024) sm[e] = 0;
  __syncthreads();
  const int p = blockIdx.x * 1024 + threadIdx.x, e = p < P ? idx[p] : E;
  if (e < E) atomicAdd(&sm[e], 1);
  __syncthreads();
  for (int i = threadIdx.x; i < E; i += 1024) hist[(int64_t)blockIdx.x * E + i] = sm[i];
}

__global__ __launch_bounds__(1024) void moe_place_kernel(const int* __restrict__ idx, int P, int E, int maxt,
                                                         const int* __restrict__ hist, int* __restrict__ meta,
                                                         int* __restrict__ order, int* __restrict__ place, int tile_rows, int tall) {
  extern __shared__ int sm[];  // cnt[E], cur[E], before[E]
  int* cnt = sm;
  int* cur = sm + E;
  int* before = sm + 2 * E;
  const int p = blockIdx.x * 1024 + threadIdx.x, e = p < P ? idx[p] : E;
  for (int i = threadIdx.x; i < E; i += 1024) cnt[i] = before[i] = 0;
  __syncthreads();
  const int n = gridDim.x * E, own = blockIdx.x * E;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const int c = hist[i];
    if (c == 0) continue;
    atomicAdd(&cnt[i % E], c);
    if (i < own) atomicAdd(&before[i % E], c);
  }
  __syncthreads();
  if (threadIdx.x < 64) group_scan(cnt, cur, E, maxt, tile_rows, blockIdx.x == 0 ? meta : nullptr, tall);
  __syncthreads();
  if (p >= P) return;
  int o = -1;
  if (e < E) {
    o = cur[e] + atomicAdd(&before[e], 1);
    order[o] = p;
  }
  place[p] = o;
}

// blocks > 1: workgroups of 1024 pairs, and `meta` has room for blocks * E counts behind its 2 + E + 2 * maxt numbers (tall: one more, the
// tiles of more than half of their rows, which stand first in the list)
void launch_moe_group(const void* idx, int P, int E, int maxt, void* meta, void* order, void* place, int tile_rows, int blocks,
                      int tall, hipStream_t st) {
  if (P == 0) return;
  if (tile_rows <= 0) throw std::runtime_error("moe_group: tile rows");
  if (E > 4096) throw std::runtime_error("moe_group: more than 4096 experts");
  if (blocks > 1) {
    if (blocks != (P + 1023) / 1024 || (int64_t)blocks * E > 0x7fffffff) throw std::runtime_error("moe_group: workgroups of 1024 pairs");
    int* hist = (int*)meta + 2 + E + 2 * (int64_t)maxt + (tall ? 1 : 0);
    moe_count_kernel<<<blocks, 1024, E * sizeof(int), st>>>((const int*)idx, P, E, hist);
    HIP_CHECK_LAUNCH();
    moe_place_kernel<<<blocks, 1024, 3 * E * sizeof(int), st>>>((const int*)idx, P, E, maxt, hist, (int*)meta, (int*)order,
                                                                (int*)place, tile_rows, tall);
    HIP_CHECK_LAUNCH();
    return;
  }
  moe_group_kernel<<<1, 1024, 2 * E * sizeof(int), st>>>((const int*)idx, P, E, maxt, (int*)meta, (int*)order,
                                                          (int*)place, tile_rows, tall);
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ grouped GEMMs
// (wg null: experts without a gate, act = gelu(up), the error-function form)
// grid (ceil(F / 64), maxt): tile y of the list covers sorted rows [row0, min(row0 + 64, off[e + 1])) of expert e.
template <typename T>
__global__ __launch_bounds__(256) void moe_gate_up_kernel(const T* __restrict__ h, int64_t ldh,
                                                          const T* __restrict__ wg, const T* __restrict__ wu,
                                                          const int* __restrict__ meta, const int* __restrict__ order,
                                                          T* __restrict__ act, int E, int maxt, int top, int F, int K,
                                                          float limit, float alpha, const float* __restrict__ pw,
                                                          int silu) {
  __shared__ float As[TV_BK][TV_LD];
  __shared__ float Gs[TV_BK][TV_LD];
  __shared__ float Us[TV_BK][TV_LD];
  if ((int)blockIdx.y >= meta[0]) return;
  const int* off = meta + 1;
  const int e = meta[1 + (E + 1) + blockIdx.y];
  const int row0 = meta[1 + (E + 1) + maxt + blockIdx.y];
  const int rows = min(TV_BM, off[e + 1] - row0);
  const int n0 = blockIdx.x * TV_BN;
  const int tid = threadIdx.x;
  const T* G = wg ? wg + (int64_t)e * F * K : nullptr;
  const T* U = wu + (int64_t)e * F * K;
  const int r = tid >> 2, kq = (tid & 3) * 4;
  const T* arow = r < rows ? h + (int64_t)(order[row0 + r] / top) * ldh : nullptr;
  const int n = n0 + r;
  float ag[4][4] = {}, au[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += TV_BK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + kq + i;
      const bool kin = k < K;
      As[kq + i][r] = (arow && kin) ? El<T>::ld(arow + k) : 0.f;
      Gs[kq + i][r] = (G && n < F && kin) ? El<T>::ld(G + (int64_t)n * K + k) : 0.f;
      Us[kq + i][r] = (n < F && kin) ? El<T>::ld(U + (int64_t)n * K + k) : 0.f;
    }
    __syncthreads();
    tv_mac(ag, As, Gs, tid);
    tv_mac(au, As, Us, tid);
    __syncthreads();
  }
  const int tx = tid & 15, ty = tid >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = ty * 4 + i;
    if (m >= rows) continue;
    const float sw = pw ? pw[order[row0 + m]] : 1.0f;  // the pair's weight on the expert's input
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int f = n0 + tx * 4 + j;
      if (f >= F) continue;
      const float v = wg ? glu_value(ag[i][j] * sw, au[i][j] * sw, limit, alpha, silu) : gelu_erf(au[i][j] * sw);
      El<T>::st(act + (int64_t)(row0 + m) * F + f, v);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void moe_down_kernel(const T* __restrict__ act, const T* __restrict__ wd,
                                                       const int* __restrict__ meta, float* __restrict__ y, int E,
                                                       int maxt, int N, int F) {
  __shared__ float As[TV_BK][TV_LD];
  __shared__ float Bs[TV_BK][TV_LD];
  if ((int)blockIdx.y >= meta[0]) return;
  const int* off = meta + 1;
  const int e = meta[1 + (E + 1) + blockIdx.y];
  const int row0 = meta[1 + (E + 1) + maxt + blockIdx.y];
  const int rows = min(TV_BM, off[e + 1] - row0);
  const int n0 = blockIdx.x * TV_BN;
  const int tid = threadIdx.x;
  const T* W = wd + (int64_t)e * N * F;
  const int r = tid >> 2, kq = (tid & 3) * 4;
  const T* arow = r < rows ? act + (int64_t)(row0 + r) * F : nullptr;
  const int n = n0 + r;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < F; k0 += TV_BK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + kq + i;
      const bool kin = k < F;
      As[kq + i][r] = (arow && kin) ? El<T>::ld(arow + k) : 0.f;
      Bs[kq + i][r] = (n < N && kin) ? El<T>::ld(W + (int64_t)n * F + k) : 0.f;
    }
    __syncthreads();
    tv_mac(acc, As, Bs, tid);
    __syncthreads();
  }
  const int tx = tid & 15, ty = tid >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = ty * 4 + i;
    if (m >= rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + tx * 4 + j;
      if (c < N) y[(int64_t)(row0 + m) * N + c] = acc[i][j];
    }
  }
}

void launch_moe_gate_up(const void* h, int64_t ldh, const void* wg, const void* wu, const void* meta,
                        const void* order, void* act, int E, int maxt, int top, int F, int K, float limit,
                        float alpha, int dt, const void* pw, int silu, hipStream_t st) {
  if (maxt <= 0) return;
  if (maxt > 65535) throw std::runtime_error("moe_gate_up: too many row tiles");
  dim3 g((F + TV_BN - 1) / TV_BN, maxt);
  DISPATCH_T(dt, T, (moe_gate_up_kernel<T><<<g, 256, 0, st>>>((const T*)h, ldh, (const T*)wg, (const T*)wu,
                                                               (const int*)meta, (const int*)order, (T*)act, E, maxt,
                                                               top, F, K, limit, alpha, (const float*)pw, silu)));
  HIP_CHECK_LAUNCH();
}

void launch_moe_down(const void* act, const void* wd, const void* meta, void* y, int E, int maxt, int N, int F,
                     int dt, hipStream_t st) {
  if (maxt <= 0) return;
  if (maxt > 65535) throw std::runtime_error("moe_down: too many row tiles");
  dim3 g((N + TV_BN - 1) / TV_BN, maxt);
  DISPATCH_T(dt, T, (moe_down_kernel<T><<<g, 256, 0, st>>>((const T*)act, (const T*)wd, (const int*)meta, (float*)y,
                                                            E, maxt, N, F)));
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ combine
template <typename T>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ y, const int* __restrict__ place,
                                                          const float* __restrict__ wts, const T* __restrict__ shared_,
                                                          int64_t lds_, float* __restrict__ out, int N, int top,
                                                          const T* __restrict__ ident, int64_t ldi,
                                                          const float* __restrict__ sw) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < N; c += blockDim.x) {
    float a = 0.f;
    for (int j = 0; j < top; ++j) {
      const int pl = place[(int64_t)t * top + j];
      const float e = pl >= 0 ? y[(int64_t)pl * N + c] : (ident ? El<T>::ld(ident + (int64_t)t * ldi + c) : 0.f);
      a = fmaf(wts ? wts[(int64_t)t * top + j] : 1.0f, e, a);
    }
    if (shared_) a = fmaf(sw ? sw[t] : 1.0f, El<T>::ld(shared_ + (int64_t)t * lds_ + c), a);
    out[(int64_t)t * N + c] = a;
  }
}

void launch_moe_combine(const void* y, const void* place, const void* wts, const void* shared_, int64_t lds_,
                        void* out, int T_, int N, int top, int dt, const void* ident, int64_t ldi, const void* sw,
                        hipStream_t st) {
  if (T_ == 0) return;
  DISPATCH_T(dt, T, (moe_combine_kernel<T><<<T_, 256, 0, st>>>((const float*)y, (const int*)place, (const float*)wts,
                                                                (const T*)shared_, lds_, (float*)out, N, top,
                                                                (const T*)ident, ldi, (const float*)sw)));
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ dense GLU
// out[t, f] = glu(gu[t, f], gu[t, F + f])
template <typename T>
__global__ __launch_bounds__(256) void glu_clamp_kernel(const T* __restrict__ gu, int64_t ldg, T* __restrict__ out,
                                                        int64_t ldo, int F, float limit, float alpha) {
  const int t = blockIdx.x;
  const T* g = gu + (int64_t)t * ldg;
  for (int f = threadIdx.x; f < F; f += blockDim.x)
    El<T>::st(out + (int64_t)t * ldo + f, glu_clamped(El<T>::ld(g + f), El<T>::ld(g + F + f), limit, alpha));
}

void launch_glu_clamp(const void* gu, int64_t ldg, void* out, int64_t ldo, int T_, int F, float limit, float alpha,
                      int dt, hipStream_t st) {
  if (T_ == 0) return;
  DISPATCH_T(dt, T, (glu_clamp_kernel<T><<<T_, 256, 0, st>>>((const T*)gu, ldg, (T*)out, ldo, F, limit, alpha)));
  HIP_CHECK_LAUNCH();
}
