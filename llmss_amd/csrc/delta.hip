// The gated delta rule in the two forms that carry a serving step, beside the token-by-token walk of recurrent.hip. Per head,
// with unit vectors k, q (q also times dim^-1/2), write strength beta = sigmoid(b) and decay g = exp(-exp(A_log) softplus(a +
// dt_bias)):   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//
//   delta_step:   steps of single rows. One workgroup per (sequence, head): the state is read once into registers and written
//                 once; S^T k and S^T q come from the same pass (o = g S^T q + (k . q) u), then the update, the per-head norm
//                 and the output gate.
//   delta_chunk:  portions of bf16 rows on the matrix cores, 64 tokens at a time. With b_t the sum of the log decays from the
//                 chunk's start to t and S_0 the state before it, the u of a chunk solve a unit lower triangular system,
//                   (I + L) U = beta (V - e^b K S_0),   L_ts = beta_t e^(b_t - b_s) k_t . k_s  (s < t)
//                   O = e^b Q S_0 + P U,                P_ts = e^(b_t - b_s) q_t . k_s         (s <= t)
//                   S_C = e^(b_C) S_0 + sum_s e^(b_C - b_s) k_s u_s^T
//                 What does not depend on the state - X = (I + L)^-1 diag(beta), P and the tokens' factors - is formed for all
//                 chunks side by side (delta_prep); the walk over the chunks is matrix products alone. The projections' q, k, v
//                 are exact in bf16 and enter unnormed, the norms being factors of rows and columns; every fp32 factor (S, U,
//                 X, P) enters as value + remainder, two bf16 numbers, and sums and the state itself stay fp32. The inverse is
//                 taken in fp32: 16 x 16 diagonal blocks by substitution, the blocks below by fp32 matrix instructions.
#include "anytype.h"
#include "chunk_rows.h"

#include <type_traits>

// ------------------------------------------------------------------------------------------------ single rows
struct DeltaStepArgs {
  const void* q;  // [T, ldq]: head group's query at q + (h / rep) * dim
  const void* k;
  const void* v;
  int64_t ldq, ldk, ldv;
  const void* a;
  const void* b;
  int64_t ldab;
  const float* A_log;
  const float* dt_bias;
  float* S;  // [slots, H, dim, vdim]
  const int* cu;
  const int* ctx;
  const int* sslots;
  const void* gate;
  int64_t ldg;
  const void* w;  // [vdim]
  float eps, scale;
  void* y;
  int64_t ldy;
  int H, G, dim, vdim;
};

// Bound by the state's bytes, read and written once, past the caches' replacement: 26.6 -> 23.5 us, and what follows finds its operands there (a
// step of 64 sequences 1.04 times as fast, with the loads alone 1.02). So it is for states of any size: chains of 16 and 24 layers, each this and a
// product of its rows, 1 - 64 sequences of 8 - 32 heads of 128 x 128 (0.5 - 128 MB a layer) 0.82 - 0.996 of the time. fp32 rows (TQ) beside bf16 projections, 64 sequences x 16 heads of 128 x
// 128: 29 us against the walk's 117.
// U: state rows per thread; a thread holds U rows x 4 columns of the state. TQ: storage of q, k, v; T: of everything else
template <typename TQ, typename T, int U>
__global__ __launch_bounds__(512) void delta_step_kernel(DeltaStepArgs A) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float red[32];
  const int h = blockIdx.x, bq = blockIdx.y, tid = threadIdx.x, nthr = blockDim.x;
  const int dim = A.dim, vdim = A.vdim, H = A.H, gq = h / (H / A.G);
  const int t = A.cu[bq], slot = A.sslots[bq], pos = A.ctx[bq] - 1;
  T* yr = (T*)A.y + (int64_t)t * A.ldy + (int64_t)h * vdim;
  if (slot < 0 || pos < 0) {
    for (int c = tid; c < vdim; c += nthr) El<T>::st(yr + c, 0.f);
    return;
  }
  float* qs = sm;                       // [dim]
  float* ks = qs + dim;                 // [dim]
  float* us = sm + ((2 * dim + 3) & ~3);  // [vdim] u
  float* pk = us + vdim;                // [row groups][vdim] parts of S^T k, then o in row 0
  const int ncg = vdim >> 2, RG = nthr / ncg, cg = tid % ncg, rg = tid / ncg;
  float* pq = pk + (int64_t)RG * vdim;
  // thread (rg, cg): columns 4 cg .. 4 cg + 3 of the state rows rg, rg + RG, ...
  float* sp = A.S + (((int64_t)slot * H + h) * dim) * (int64_t)vdim + 4 * cg;
  f32x4 s[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = rg + u * RG;
    s[u] = (pos > 0 && rg < RG && r < dim) ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(sp + (int64_t)r * vdim)) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float zb = El<T>::ld((const T*)A.b + (int64_t)t * A.ldab + h);
  const float za = El<T>::ld((const T*)A.a + (int64_t)t * A.ldab + h) + A.dt_bias[h];
  const float beta = 1.0f / (1.0f + expf(-zb));
  const float g = expf(-expf(A.A_log[h]) * (za > 20.f ? za : log1pf(expf(za))));
  const TQ* qr = (const TQ*)A.q + (int64_t)t * A.ldq + (int64_t)gq * dim;
  const TQ* kr = (const TQ*)A.k + (int64_t)t * A.ldk + (int64_t)gq * dim;
  float qq = 0.f, kk = 0.f, kq = 0.f;
  for (int d = tid; d < dim; d += nthr) {
    const float qd = El<TQ>::ld(qr + d), kd = El<TQ>::ld(kr + d);
    qs[d] = qd;
    ks[d] = kd;
    qq = fmaf(qd, qd, qq);
    kk = fmaf(kd, kd, kk);
    kq = fmaf(kd, qd, kq);
  }
  const f32x2 s2 = block_sum2(qq, kk, red);
  kq = block_sum(kq, red);  // (the barriers also make qs, ks visible)
  const float qn = 1.0f / (sqrtf(s2[0] + 1e-6f) * sqrtf((float)dim)), kn = 1.0f / sqrtf(s2[1] + 1e-6f);
  if (rg < RG) {
    f32x4 ak = {0.f, 0.f, 0.f, 0.f}, aq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = min(rg + u * RG, dim - 1);  // (rows past the state hold zeros)
      const float kd = ks[r], qd = qs[r];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ak[i] = fmaf(s[u][i], kd, ak[i]);
        aq[i] = fmaf(s[u][i], qd, aq[i]);
      }
    }
    *reinterpret_cast<f32x4*>(pk + (int64_t)rg * vdim + 4 * cg) = ak;
    *reinterpret_cast<f32x4*>(pq + (int64_t)rg * vdim + 4 * cg) = aq;
  }
  __syncthreads();
  float ss = 0.f;
  for (int c = tid; c < vdim; c += nthr) {
    float a = 0.f, o = 0.f;
    for (int r = 0; r < RG; ++r) {
      a += pk[r * vdim + c];
      o += pq[r * vdim + c];
    }
    const float v = El<TQ>::ld((const TQ*)A.v + (int64_t)t * A.ldv + (int64_t)h * vdim + c);
    const float u = beta * (v - g * kn * a);
    us[c] = u;
    o = g * qn * o + kq * kn * qn * u;
    pk[c] = o;  // (row 0 of the parts at this column: read by this thread alone)
    ss = fmaf(o, o, ss);
  }
  ss = block_sum(ss, red);  // (its barriers make us visible)
  if (rg < RG) {
    const f32x4 u4 = *reinterpret_cast<const f32x4*>(us + 4 * cg);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = rg + u * RG;
      if (r < dim) {
        const float kd = ks[r] * kn;
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = fmaf(g, s[u][i], kd * u4[i]);
        __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(sp + (int64_t)r * vdim));
      }
    }
  }
  const float inv = A.scale / sqrtf(ss / (float)vdim + A.eps);
  const T* gr = (const T*)A.gate + (int64_t)t * A.ldg + (int64_t)h * vdim;
  for (int c = tid; c < vdim; c += nthr) {
    const float z = El<T>::ld(gr + c);
    El<T>::st(yr + c, pk[c] * inv * El<T>::ld((const T*)A.w + c) * (z / (1.0f + expf(-z))));
  }
}

static int delta_step_threads(int dim, int vdim) {
  if (vdim % 4 || vdim < 4 || vdim > 1024 || dim < 1 || dim > 512) return 0;
  for (int th = 256; th <= 512; th *= 2)
    if (th >= vdim / 4 && (dim + th / (vdim / 4) - 1) / (th / (vdim / 4)) <= 16) return th;
  return 0;
}
bool delta_step_ok(int dim, int vdim) { return delta_step_threads(dim, vdim) > 0; }

// B sequences of one row each
void launch_delta_step(const void* q, const void* k, const void* v, int64_t ldq, int64_t ldk, int64_t ldv, const void* a,
                       const void* b, int64_t ldab, const void* A_log, const void* dt_bias, void* S, const void* cu,
                       const void* ctx, const void* sslots, const void* gate, int64_t ldg, const void* w, float eps,
                       float scale, void* y, int64_t ldy, int B, int H, int G, int dim, int vdim, int dq, int dt, hipStream_t st) {
  if (B == 0) return;
  const int th = delta_step_threads(dim, vdim);
  if (!th || B > 65535 || G < 1 || H % G) throw std::runtime_error("delta_step: shape");
  if ((uintptr_t)S & 15) throw std::runtime_error("delta_step: the state must be 16-byte aligned");
  DeltaStepArgs A{q, k, v, ldq, ldk, ldv, a, b, ldab, (const float*)A_log, (const float*)dt_bias, (float*)S, (const int*)cu,
                  (const int*)ctx, (const int*)sslots, gate, ldg, w, eps, scale, y, ldy, H, G, dim, vdim};
  const int RG = th / (vdim / 4), U = (dim + RG - 1) / RG;
  const size_t lds = ((size_t)2 * dim + 4 + vdim + (size_t)2 * RG * vdim) * 4;
  dim3 g(H, B);
  if (dq == 0 && dt != 0) throw std::runtime_error("delta_step: 16-bit rows beside 32-bit projections");
#define LAUNCH_DS(TQ_, T_)                                                       \
  do {                                                                           \
    if (U <= 4) delta_step_kernel<TQ_, T_, 4><<<g, th, lds, st>>>(A);            \
    else if (U <= 8) delta_step_kernel<TQ_, T_, 8><<<g, th, lds, st>>>(A);       \
    else delta_step_kernel<TQ_, T_, 16><<<g, th, lds, st>>>(A);                  \
  } while (0)
  if (dq == 0) LAUNCH_DS(bf16_t, bf16_t);
  else if (dt == 0) LAUNCH_DS(float, bf16_t);
  else LAUNCH_DS(float, float);
#undef LAUNCH_DS
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ portions
struct DeltaChunkArgs {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  int64_t ldq, ldk, ldv;
  const bf16_t* a;
  const bf16_t* b;
  int64_t ldab;
  const float* A_log;
  const float* dt_bias;
  float* S;
  const int* cu;
  const int* ctx;
  const int* sslots;
  float* out;  // [T, H * vdim]
  bf16_t* X;   // [4][T, H, 64]: X value, X remainder, P value, P remainder; row t of its chunk
  int64_t mat;  // numbers per matrix
  f32x4* aux;  // [T, H] (e^b |k|^-1, e^b |q|^-1 dim^-1/2, e^(b_C - b) |k|^-1, e^(b_C))
  int H, G, dim, vdim;
};

__device__ __forceinline__ void split2(float x, bf16_t& hi, bf16_t& lo) {
  hi = f2bf(x);
  lo = f2bf(x - bf2f(hi));
}

// A lane's column of the state, rows r0 + 16 kt + i; zeros where there is none. (All loads first.)
template <int N>
__device__ __forceinline__ void load_state(f32x4 (&S)[N], bool cont, const float* sp, int r0, int dim, int vdim, int col) {
#pragma unroll
  for (int kt = 0; kt < N; ++kt) S[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (!cont) return;
  const float* const p = sp + min(col, vdim - 1);
#pragma unroll
  for (int kt = 0; kt < N; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[kt][i] = p[(int64_t)min(r0 + 16 * kt + i, dim - 1) * vdim];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int kt = 0; kt < N; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[kt][i] = r0 + 16 * kt + i < dim && col < vdim ? S[kt][i] : 0.f;
}

constexpr int prep_kq_bytes(int kt) {  // K and Q rows, or P (value, remainder) and the fp32 inverse
  return 2 * 64 * (16 * kt + 8) * 2 > 2 * 64 * 72 * 2 + 64 * 68 * 4 ? 2 * 64 * (16 * kt + 8) * 2 : 2 * 64 * 72 * 2 + 64 * 68 * 4;
}

// (I + L)^-1 of a 64 x 64 matrix in LDS (4 waves; the blocks of X above the diagonal hold zeros already)
__device__ __forceinline__ void lower_inverse(const float* Ls, float* Xs, const int LDL, int w, int li, int g) {
  // wave w its 16 x 16 diagonal block by substitution, a column per lane (four copies of each)
  {
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) x[t] = t == li ? 1.0f : 0.f;
#pragma unroll
    for (int t = 1; t < 16; ++t) {
      const float* lr = &Ls[(16 * w + t) * LDL + 16 * w];
      float acc = 0.f, acc2 = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) {
        if (s & 1) acc2 = fmaf(lr[s], x[s], acc2);
        else acc = fmaf(lr[s], x[s], acc);
      }
      x[t] -= acc + acc2;
    }
#pragma unroll
    for (int t = 0; t < 16; ++t)
      if ((t >> 2) == g) Xs[(16 * w + t) * LDL + 16 * w + li] = x[t];
  }
  // the blocks below, a diagonal at a time: X_ij = -X_ii sum_{j <= m < i} L_im X_mj
#pragma unroll
  for (int lev = 1; lev < 4; ++lev) {
    __syncthreads();
    const int bi = w + lev, bj = w;
    if (bi < 4) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f}, o = {0.f, 0.f, 0.f, 0.f};
      for (int m = bj; m < bi; ++m) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          z = __builtin_amdgcn_mfma_f32_16x16x4f32(Ls[(16 * bi + li) * LDL + 16 * m + 4 * g + i],
                                                   Xs[(16 * m + 4 * g + i) * LDL + 16 * bj + li], z, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) z[i] = fabsf(z[i]) <= FLT_MAX ? z[i] : 0.f;  // (rows that are NaN in any case: not into those above)
#pragma unroll
      for (int i = 0; i < 4; ++i)  // (the accumulator's rows 4 g + i are the second operand as they stand)
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(Xs[(16 * bi + li) * LDL + 16 * bi + 4 * g + i], z[i], o, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) Xs[(16 * bi + 4 * g + i) * LDL + 16 * bj + li] = -o[i];
    }
  }
  __syncthreads();
}

// Workgroup (chunk of a portion, head, sequence), 4 waves
template <int KT>
__global__ __launch_bounds__(256) void delta_prep_kernel(DeltaChunkArgs A) {
  constexpr int C = 64, DKP = 16 * KT, LDK = DKP + 8, LDP = 64 + 8, LDL = 64 + 4;
  constexpr int KQ = prep_kq_bytes(KT);  // the rows' region; once their products are taken P and the inverse lie there
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* Ks = reinterpret_cast<bf16_t*>(smem);
  bf16_t* Qs = Ks + C * LDK;
  bf16_t* Ph = reinterpret_cast<bf16_t*>(smem);
  bf16_t* Pl = Ph + C * LDP;
  float* Xs = reinterpret_cast<float*>(Pl + C * LDP);     // [64][LDL]
  float* Ls = reinterpret_cast<float*>(smem + KQ);        // [64][LDL]
  float* bs = Ls + C * LDL;                               // [64] sum of the log decays
  float* be = bs + C;                                  // [64] write strength
  float* nk = be + C;                                  // [64] 1 / |k|
  float* nq = nk + C;                                  // [64] dim^-1/2 / |q|
  const int b = blockIdx.z, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int t0 = A.cu[b], qlen = A.cu[b + 1] - t0, j0 = blockIdx.x * C;
  if (j0 >= qlen || A.sslots[b] < 0 || A.ctx[b] <= 0) return;
  const int nt = min(C, qlen - j0), dim = A.dim, H = A.H, gq = h / (H / A.G);
  constexpr int CHK = DKP / 8, NK = C * CHK / 256;
  static_assert((C * CHK) % 256 == 0, "whole 16-byte pieces per thread");
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // (all loads first, from the nearest place that is there: behind a condition each was waited for before the next, a memory's latency each)
  u16x8 rk[NK], rq[NK];
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 8;
    const int64_t tt = t0 + j0 + min(r, nt - 1), at = (int64_t)gq * dim + (d < dim ? d : 0);
    rk[j] = *reinterpret_cast<const u16x8*>(A.k + tt * A.ldk + at);
    rq[j] = *reinterpret_cast<const u16x8*>(A.q + tt * A.ldq + at);
  }
  const int64_t tab = (int64_t)(t0 + j0 + min(lane, nt - 1)) * A.ldab + h;
  const bf16_t ra = A.a[tab], rb = A.b[tab];
  const float alog = A.A_log[h], dtb = A.dt_bias[h];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 8;
    const bool in = r < nt && d < dim;
    *reinterpret_cast<u16x8*>(&Ks[r * LDK + d]) = in ? rk[j] : zero8;
    *reinterpret_cast<u16x8*>(&Qs[r * LDK + d]) = in ? rq[j] : zero8;
  }
  if (w == 0) {  // the tokens' decays and write strengths
    const bool in = lane < nt;
    const float z = bf2f(ra) + dtb;
    float F = in ? -expf(alog) * (z > 20.f ? z : log1pf(expf(z))) : 0.f;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float x = __shfl_up(F, o, 64);
      if (lane >= o) F += x;
    }
    bs[lane] = F;
    be[lane] = in ? 1.0f / (1.0f + expf(-bf2f(rb))) : 0.f;
  }
  __syncthreads();
  {  // norms: four neighbouring lanes per row
    const int r = tid >> 2, part = tid & 3;
    float kk = 0.f, qq = 0.f;
    for (int d = part * 8; d < DKP; d += 32) {
      const u16x8 x = *reinterpret_cast<const u16x8*>(&Ks[r * LDK + d]), y = *reinterpret_cast<const u16x8*>(&Qs[r * LDK + d]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        kk = fmaf(bf2f(x[i]), bf2f(x[i]), kk);
        qq = fmaf(bf2f(y[i]), bf2f(y[i]), qq);
      }
    }
    kk += __shfl_xor(kk, 1, 64);
    kk += __shfl_xor(kk, 2, 64);
    qq += __shfl_xor(qq, 1, 64);
    qq += __shfl_xor(qq, 2, 64);
    if (part == 0) {
      nk[r] = 1.0f / sqrtf(kk + 1e-6f);
      nq[r] = 1.0f / (sqrtf(qq + 1e-6f) * sqrtf((float)dim));
    }
  }
  __syncthreads();
  // wave w: the products of its 16 tokens (rows) with the keys of the blocks up to its own (columns)
  {
    f32x4 pk[4], pq[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) pk[ct] = pq[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KT / 2; ++ks) {
      const s16x8 ka = *reinterpret_cast<const s16x8*>(&Ks[(16 * w + li) * LDK + 32 * ks + 8 * g]);
      const s16x8 qa = *reinterpret_cast<const s16x8*>(&Qs[(16 * w + li) * LDK + 32 * ks + 8 * g]);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        if (ct > w) continue;
        const s16x8 kb = *reinterpret_cast<const s16x8*>(&Ks[(16 * ct + li) * LDK + 32 * ks + 8 * g]);
        pk[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, kb, pk[ct], 0, 0, 0);
        pq[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa, kb, pq[ct], 0, 0, 0);
      }
    }
    __syncthreads();  // every wave has read its rows
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int s = 16 * ct + li;
      const float bsv = bs[s], nks = nk[s];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * w + 4 * g + i;
        const float e = s <= t ? expf(bs[t] - bsv) * nks : 0.f;
        Ls[t * LDL + s] = s < t ? e * be[t] * nk[t] * pk[ct][i] : 0.f;
        split2(s <= t ? e * nq[t] * pq[ct][i] : 0.f, Ph[t * LDP + s], Pl[t * LDP + s]);
        if (ct > w) Xs[t * LDL + s] = 0.f;  // the blocks of the inverse above the diagonal
      }
    }
  }
  __syncthreads();
  lower_inverse(Ls, Xs, LDL, w, li, g);
  const int64_t row = (int64_t)(t0 + j0) * H + h;
  for (int e = tid; e < C * 8; e += 256) {
    const int r = e >> 3, s0 = (e & 7) * 8;
    if (r >= nt) continue;
    u16x8 xh, xl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      bf16_t hi, lo;
      split2(Xs[r * LDL + s0 + i] * be[s0 + i], hi, lo);
      xh[i] = hi;
      xl[i] = lo;
    }
    bf16_t* dst = A.X + (row + (int64_t)r * H) * 64 + s0;
    *reinterpret_cast<u16x8*>(dst) = xh;
    *reinterpret_cast<u16x8*>(dst + A.mat) = xl;
    *reinterpret_cast<u16x8*>(dst + 2 * A.mat) = *reinterpret_cast<const u16x8*>(&Ph[r * LDP + s0]);
    *reinterpret_cast<u16x8*>(dst + 3 * A.mat) = *reinterpret_cast<const u16x8*>(&Pl[r * LDP + s0]);
  }
  if (tid < nt) {
    const float e = expf(bs[tid]), bc = bs[C - 1];
    A.aux[row + (int64_t)tid * H] = f32x4{e * nk[tid], e * nq[tid], expf(bc - bs[tid]) * nk[tid], expf(bc)};
  }
}

// Workgroup (head, block of 64 value columns, sequence), 4 waves, the portion's chunks in order. A wave owns 16 value columns:
// its part of the state lives in registers in the accumulator layout (lane (li, g): column li, rows 16 tile + 4 g + i), whose
// rows are, without any exchange, the k-slots (8 g + j -> row 4 g + j of tile 2 ks, j < 4, or 4 g + j - 4 of tile 2 ks + 1) of
// the second operand of the next product - and so are V - e^b K S_0 and U over the tokens. The next chunk's rows and
// matrices are fetched into registers while this one is computed; nothing inside a chunk waits for another wave.
template <int KT>
__global__ __launch_bounds__(256) void delta_chunk_kernel(DeltaChunkArgs A) {
  constexpr int C = 64, DKP = 16 * KT, LDK = DKP + 8, LDP = 64 + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* Qs = reinterpret_cast<bf16_t*>(smem);
  bf16_t* Ks = Qs + C * LDK;
  bf16_t* Ms = Ks + C * LDK;                          // [4][64][LDP]
  f32x4* ax = reinterpret_cast<f32x4*>(Ms + 4 * C * LDP);  // [64]
  const int h = blockIdx.x, b = gridDim.z - 1 - blockIdx.z;
  const int dim = A.dim, vdim = A.vdim, H = A.H, gq = h / (H / A.G);
  const int t0 = A.cu[b], qlen = A.cu[b + 1] - t0, slot = A.sslots[b], ctx = A.ctx[b];
  if (qlen <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int col = blockIdx.y * 64 + 16 * w + li, colc = min(col, vdim - 1);
  float* outp = A.out + (int64_t)t0 * H * vdim + (int64_t)h * vdim + col;
  if (slot < 0 || ctx <= 0) {
    if (g == 0 && col < vdim)
      for (int j = 0; j < qlen; ++j) outp[(int64_t)j * H * vdim] = 0.f;
    return;
  }
  const bool cont = ctx > qlen;  // continues an earlier portion
  f32x4 S[KT];
  float* sp = A.S + (((int64_t)slot * H + h) * dim) * (int64_t)vdim;
  load_state(S, cont, sp, 4 * g, dim, vdim, col);
  constexpr int CHK = DKP / 8, NK = C * CHK / 256;
  u16x8 rq[NK], rk[NK], rm[8];
  uint32_t rv[16];  // (words: two numbers to a register wait for both)
  f32x4 ra = {0.f, 0.f, 0.f, 0.f};
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  auto fetch = [&](int j0) {  // (as in delta_chunk32)
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 8;
      const int64_t tt = t0 + min(j0 + r, qlen - 1), at = (int64_t)gq * dim + (d < dim ? d : 0);
      rq[j] = *reinterpret_cast<const u16x8*>(A.q + tt * A.ldq + at);
      rk[j] = *reinterpret_cast<const u16x8*>(A.k + tt * A.ldk + at);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = tid + 256 * (j & 1), r = c >> 3, s0 = (c & 7) * 8;
      rm[j] = *reinterpret_cast<const u16x8*>(A.X + (j >> 1) * A.mat + ((int64_t)(t0 + min(j0 + r, qlen - 1)) * H + h) * 64 + s0);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {  // token 16 (j / 4) + 4 g + j % 4 at this lane's column
      const int r = j0 + 16 * (j >> 2) + 4 * g + (j & 3);
      rv[j] = A.v[(int64_t)(t0 + min(r, qlen - 1)) * A.ldv + (int64_t)h * vdim + colc];
    }
    ra = A.aux[(int64_t)(t0 + min(j0 + lane, qlen - 1)) * H + h];
  };
  fetch(0);
  for (int j0 = 0; j0 < qlen; j0 += C) {
    const int nt = min(C, qlen - j0);
    __syncthreads();  // the previous chunk's readers are done
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 8;
      const bool in = r < nt && d < dim;
      *reinterpret_cast<u16x8*>(&Qs[r * LDK + d]) = in ? rq[j] : zero8;
      *reinterpret_cast<u16x8*>(&Ks[r * LDK + d]) = in ? rk[j] : zero8;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = tid + 256 * (j & 1);
      *reinterpret_cast<u16x8*>(&Ms[(j >> 1) * C * LDP + (c >> 3) * LDP + (c & 7) * 8]) = (c >> 3) < nt ? rm[j] : zero8;
    }
    if (w == 0) ax[lane] = ra;
    f32x4 u[4];  // first V, then V - e^b K S_0
#pragma unroll
    for (int j = 0; j < 16; ++j) u[j >> 2][j & 3] = bf2f((bf16_t)rv[j]);
    __syncthreads();
    if (j0 + C < qlen) fetch(j0 + C);
    // K S_0 and Q S_0 for this wave's columns
    f32x4 o[4], ksv[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) o[rt] = ksv[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KT / 2; ++ks) {
      s16x8 sh, sl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        bf16_t hi, lo;
        split2(S[2 * ks + (j >> 2)][j & 3], hi, lo);
        sh[j] = (short)hi;
        sl[j] = (short)lo;
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const bf16_t* kp = &Ks[(16 * rt + li) * LDK + 32 * ks + 4 * g];
        const s16x4 k0 = *reinterpret_cast<const s16x4*>(kp), k1 = *reinterpret_cast<const s16x4*>(kp + 16);
        const s16x8 ka = {k0[0], k0[1], k0[2], k0[3], k1[0], k1[1], k1[2], k1[3]};
        ksv[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, sh, ksv[rt], 0, 0, 0);
        ksv[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, sl, ksv[rt], 0, 0, 0);
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const bf16_t* qp = &Qs[(16 * rt + li) * LDK + 32 * ks + 4 * g];
        const s16x4 q0 = *reinterpret_cast<const s16x4*>(qp), q1 = *reinterpret_cast<const s16x4*>(qp + 16);
        const s16x8 qa = {q0[0], q0[1], q0[2], q0[3], q1[0], q1[1], q1[2], q1[3]};
        o[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa, sh, o[rt], 0, 0, 0);
        o[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa, sl, o[rt], 0, 0, 0);
      }
    }
    f32x4 wgt[4];  // e^(b_C - b) |k|^-1 of this lane's tokens
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 x = ax[16 * rt + 4 * g + i];
        u[rt][i] = fmaf(-x[0], ksv[rt][i], u[rt][i]);
        o[rt][i] *= x[1];
        wgt[rt][i] = x[2];
      }
    const float a_all = ax[0][3];
    // the products with X and then P: operand rows 16 rt + li, the second operand in registers
    auto lower = [&](const bf16_t* m, const f32x4* x, f32x4* acc) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        s16x8 xh, xl;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          bf16_t hi, lo;
          split2(x[2 * ks + (j >> 2)][j & 3], hi, lo);
          xh[j] = (short)hi;
          xl[j] = (short)lo;
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          if (16 * rt + 15 < 32 * ks) continue;  // tokens before every token of this half
          const bf16_t* p = &m[(16 * rt + li) * LDP + 32 * ks + 4 * g];
          const s16x4 h0 = *reinterpret_cast<const s16x4*>(p), h1 = *reinterpret_cast<const s16x4*>(p + 16);
          const s16x4 l0 = *reinterpret_cast<const s16x4*>(p + C * LDP), l1 = *reinterpret_cast<const s16x4*>(p + C * LDP + 16);
          const s16x8 mh = {h0[0], h0[1], h0[2], h0[3], h1[0], h1[1], h1[2], h1[3]};
          const s16x8 ml = {l0[0], l0[1], l0[2], l0[3], l1[0], l1[1], l1[2], l1[3]};
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mh, xh, acc[rt], 0, 0, 0);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mh, xl, acc[rt], 0, 0, 0);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ml, xh, acc[rt], 0, 0, 0);
        }
      }
    };
    f32x4 U[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) U[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    lower(Ms, u, U);
    lower(Ms + 2 * C * LDP, U, o);
    // the state: K^T (w U)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[kt][i] *= a_all;
    const int tq = li >> 2, tp = li & 3;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      s16x8 vh, vl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        bf16_t hi, lo;
        split2(U[2 * ks + (j >> 2)][j & 3] * wgt[2 * ks + (j >> 2)][j & 3], hi, lo);
        vh[j] = (short)hi;
        vl[j] = (short)lo;
      }
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const bf16_t* k0 = &Ks[(32 * ks + 4 * g + tq) * LDK + 16 * kt + 4 * tp];
        const s16x4 y0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(k0));
        const s16x4 y1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(k0 + 16 * LDK));
        const s16x8 ka = {y0[0], y0[1], y0[2], y0[3], y1[0], y1[1], y1[2], y1[3]};
        S[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, vh, S[kt], 0, 0, 0);
        S[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, vl, S[kt], 0, 0, 0);
      }
    }
    if (col < vdim) {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * rt + 4 * g + i;
          if (t < nt) outp[(int64_t)(j0 + t) * H * vdim] = o[rt][i];
        }
    }
  }
  if (col < vdim) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * kt + 4 * g + i;
        if (r < dim) sp[(int64_t)r * vdim + col] = S[kt][i];
      }
  }
}

bool delta_chunk_ok(int dim, int vdim) { return dim % 8 == 0 && dim >= 8 && dim <= 256 && vdim >= 1; }

// max_qlen: rows of the longest portion; work: bf16 [4][T, H, 64]; aux: fp32 [T, H, 4]
void launch_delta_chunk(const void* q, const void* k, const void* v, int64_t ldq, int64_t ldk, int64_t ldv, const void* a,
                        const void* b, int64_t ldab, const void* A_log, const void* dt_bias, void* S, const void* cu,
                        const void* ctx, const void* sslots, void* out, void* work, void* aux, int T_, int B, int max_qlen,
                        int H, int G, int dim, int vdim, hipStream_t st) {
  if (B == 0 || max_qlen <= 0) return;
  if (!delta_chunk_ok(dim, vdim) || B > 65535 || H > 65535 || G < 1 || H % G) throw std::runtime_error("delta_chunk: shape");
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)work | (uintptr_t)aux) & 15 || (ldq | ldk) & 7)
    throw std::runtime_error("delta_chunk: rows must be 16-byte aligned");
  DeltaChunkArgs A{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldq, ldk, ldv, (const bf16_t*)a, (const bf16_t*)b,
                   ldab, (const float*)A_log, (const float*)dt_bias, (float*)S, (const int*)cu, (const int*)ctx,
                   (const int*)sslots, (float*)out, (bf16_t*)work, (int64_t)T_ * H * 64, (f32x4*)aux, H, G, dim, vdim};
  dim3 g1((max_qlen + 63) / 64, H, B), g2(H, (vdim + 63) / 64, B);
  auto lds1 = [](int kt) {
    return (size_t)prep_kq_bytes(kt) + (size_t)4 * (64 * 68 + 4 * 64);
  };
  auto lds2 = [](int kt) { return (size_t)2 * (2 * 64 * (16 * kt + 8) + 4 * 64 * 72) + (size_t)16 * 64; };
#define LAUNCH_DC(KT_)                                                                                           \
  do {                                                                                                           \
    static bool once = [] {                                                                                      \
      (void)hipFuncSetAttribute((const void*)delta_prep_kernel<KT_>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                160 * 1024);                                                                     \
      (void)hipFuncSetAttribute((const void*)delta_chunk_kernel<KT_>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                160 * 1024);                                                                     \
      return true;                                                                                               \
    }();                                                                                                         \
    (void)once;                                                                                                  \
    delta_prep_kernel<KT_><<<g1, 256, lds1(KT_), st>>>(A);                                                       \
    delta_chunk_kernel<KT_><<<g2, 256, lds2(KT_), st>>>(A);                                                      \
  } while (0)
  if (dim <= 32) LAUNCH_DC(2);
  else if (dim <= 64) LAUNCH_DC(4);
  else if (dim <= 128) LAUNCH_DC(8);
  else LAUNCH_DC(16);
#undef LAUNCH_DC
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ portions of fp32 rows
// The same two kernels for rows in 32 bits (a convolution's fp32 results), every product on the fp32 matrix instructions, the
// sums of log decays in 64 bits, X and P held in 32. Bound by the chain of chunks: 8 sequences x 16
// heads of 128 x 128 are one workgroup per CU (wave per SIMD), each 16 dependent chunks of 464 matrix instructions of 32 cycles.
// 8 x 1024 tokens: 408 us with the norm, 1615 us token by token; one sequence of 2048: 440 and 3130 us.
struct DeltaChunk32Args {
  const float* q;
  const float* k;
  const float* v;
  int64_t ldq, ldk, ldv;
  const void* a;
  const void* b;
  int64_t ldab;
  const float* A_log;
  const float* dt_bias;
  float* S;
  const int* cu;
  const int* ctx;
  const int* sslots;
  float* out;  // [T, H * vdim]
  float* X;    // [2][T, H, 64]: X, P; row t of its chunk
  int64_t mat;
  f32x4* aux;  // as above
  int H, G, dim, vdim;
};

__device__ __forceinline__ f32x4 ldv4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

constexpr int prep32_k_bytes(int kt) {  // K rows, or P and the inverse
  return 64 * (16 * kt + 4) * 4 > 2 * 64 * 68 * 4 ? 64 * (16 * kt + 4) * 4 : 2 * 64 * 68 * 4;
}

// acc += A B^T over the keys: A's row in registers (columns 16 kt + 4 g on), B's at bp (this lane's, from column 4 g on), in up to four
// chains (shorter ones round less)
template <int KT>
__device__ __forceinline__ f32x4 dot32(const f32x4* a, const float* bp) {
  constexpr int N = KT < 4 ? 2 : 4;
  f32x4 c[N];
#pragma unroll
  for (int n = 0; n < N; ++n) c[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < KT; kt += N) {
    f32x4 x[N], y[N];
#pragma unroll
    for (int n = 0; n < N; ++n) x[n] = a[kt + n], y[n] = ldv4(bp + 16 * (kt + n));
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < N; ++n) c[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[n][i], y[n][i], c[n], 0, 0, 0);
  }
  return N == 4 ? (c[0] + c[1]) + (c[N - 2] + c[N - 1]) : c[0] + c[1];
}
// A S: the state's tiles are the second operand as they stand
template <int KT>
__device__ __forceinline__ f32x4 dot32s(const f32x4 (&x)[KT], const f32x4 (&S)[KT]) {
  constexpr int N = KT < 4 ? 2 : 4;
  f32x4 c[N];
#pragma unroll
  for (int n = 0; n < N; ++n) c[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < KT; kt += N)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < N; ++n) c[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[kt + n][i], S[kt + n][i], c[n], 0, 0, 0);
  return N == 4 ? (c[0] + c[1]) + (c[N - 2] + c[N - 1]) : c[0] + c[1];
}

// Workgroup (chunk of a portion, head, sequence), 4 waves. TP: storage of a and b. Bound by its chain of stages (rows, sums, products,
// 64 steps of substitution), so by how many workgroups a CU holds: the queries stay in the registers of the wave whose rows they
// are, and 54 KB of LDS let three in where keys and queries in LDS (86 KB) left room for one. With all loads before the first use 80 -> 66 us
// (8 x 1024 tokens, 16 heads of 128), delta_prep 75 -> 60, delta_chunk 133 -> 111 (7 x 1180).
template <int KT, typename TP>
__global__ __launch_bounds__(256, 3) void delta_prep32_kernel(DeltaChunk32Args A) {
  constexpr int C = 64, DKP = 16 * KT, LDK = DKP + 4, LDL = 64 + 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* Ks = reinterpret_cast<float*>(smem);
  float* Ps = reinterpret_cast<float*>(smem);  // once the rows' products are taken
  float* Xs = Ps + C * LDL;
  float* Ls = reinterpret_cast<float*>(smem + prep32_k_bytes(KT));
  double* bs = reinterpret_cast<double*>(Ls + C * LDL);  // [64] sum of the log decays
  float* be = reinterpret_cast<float*>(bs + C);          // [64] write strength
  float* nk = be + C;                                    // [64] 1 / |k|
  float* nq = nk + C;                                    // [64] dim^-1/2 / |q|
  const int b = blockIdx.z, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int t0 = A.cu[b], qlen = A.cu[b + 1] - t0, j0 = blockIdx.x * C;
  if (j0 >= qlen || A.sslots[b] < 0 || A.ctx[b] <= 0) return;
  const int nt = min(C, qlen - j0), dim = A.dim, H = A.H, gq = h / (H / A.G);
  constexpr int CHK = DKP / 4, NK = C * CHK / 256;
  static_assert((C * CHK) % 256 == 0, "whole 16-byte pieces per thread");
  // (all loads first, as in delta_prep)
  f32x4 rk[NK];
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 4;
    rk[j] = ldv4(A.k + (int64_t)(t0 + j0 + min(r, nt - 1)) * A.ldk + (int64_t)gq * dim + (d < dim ? d : 0));
  }
  const int64_t tab = (int64_t)(t0 + j0 + min(lane, nt - 1)) * A.ldab + h;
  const TP ra = ((const TP*)A.a)[tab], rb = ((const TP*)A.b)[tab];
  const float alog = A.A_log[h], dtb = A.dt_bias[h];
  f32x4 q[KT];  // row 16 w + li, columns 16 kt + 4 g on
  {
    const float* qp = A.q + (int64_t)(t0 + j0 + min(16 * w + li, nt - 1)) * A.ldq + (int64_t)gq * dim;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) q[kt] = ldv4(qp + (16 * kt + 4 * g < dim ? 16 * kt + 4 * g : 0));
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 4;
    *reinterpret_cast<f32x4*>(&Ks[r * LDK + d]) = r < nt && d < dim ? rk[j] : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) q[kt] = 16 * w + li < nt && 16 * kt + 4 * g < dim ? q[kt] : f32x4{0.f, 0.f, 0.f, 0.f};
  if (w == 0) {  // the tokens' decays and write strengths
    const bool in = lane < nt;
    const float z = El<TP>::ld(&ra) + dtb;
    // (a decay of zero: a sum this low vanishes over a single token, and differences of equal sums stay zero)
    double F = in ? at_least((double)(-expf(alog) * (z > 20.f ? z : log1pf(expf(z)))), -1e8) : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double x = __shfl_up(F, o, 64);
      if (lane >= o) F += x;
    }
    bs[lane] = F;
    be[lane] = in ? 1.0f / (1.0f + expf(-El<TP>::ld(&rb))) : 0.f;
  }
  __syncthreads();
  {  // norms: four neighbouring lanes per row
    const int r = tid >> 2, part = tid & 3;
    float kk = 0.f, qq = 0.f;
    for (int d = part * 4; d < DKP; d += 16) {
      const f32x4 x = ldv4(&Ks[r * LDK + d]);
#pragma unroll
      for (int i = 0; i < 4; ++i) kk = fmaf(x[i], x[i], kk);
    }
    kk += __shfl_xor(kk, 1, 64);
    kk += __shfl_xor(kk, 2, 64);
    if (part == 0) nk[r] = 1.0f / sqrtf(kk + 1e-6f);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) qq = fmaf(q[kt][i], q[kt][i], qq);
    qq = xor32_sum(xor16_sum(qq));
    if (g == 0) nq[16 * w + li] = 1.0f / (sqrtf(qq + 1e-6f) * sqrtf((float)dim));
  }
  // wave w: the products of its 16 tokens (rows) with the keys of the blocks up to its own (columns)
  f32x4 pk[4], pq[4], ka[KT];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) ka[kt] = ldv4(&Ks[(16 * w + li) * LDK + 16 * kt + 4 * g]);
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    pk[ct] = pq[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (ct > w || 16 * w >= nt) continue;
    const float* kb = &Ks[(16 * ct + li) * LDK + 4 * g];
    pk[ct] = dot32<KT>(ka, kb);
    pq[ct] = dot32<KT>(q, kb);
  }
  __syncthreads();  // every wave has read its rows; the norms are written
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const int s = 16 * ct + li;
    const double bsv = bs[s];
    const float nks = nk[s];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * w + 4 * g + i;
      const float e = s <= t ? expf((float)(bs[t] - bsv)) * nks : 0.f;
      Ls[t * LDL + s] = s < t ? e * be[t] * nk[t] * pk[ct][i] : 0.f;
      Ps[t * LDL + s] = s <= t ? e * nq[t] * pq[ct][i] : 0.f;
      if (ct > w) Xs[t * LDL + s] = 0.f;  // the blocks of the inverse above the diagonal
    }
  }
  __syncthreads();
  lower_inverse(Ls, Xs, LDL, w, li, g);
  const int64_t row = (int64_t)(t0 + j0) * H + h;
  for (int e = tid; e < C * 16; e += 256) {
    const int r = e >> 4, s0 = (e & 15) * 4;
    if (r >= nt) continue;
    f32x4 x = ldv4(&Xs[r * LDL + s0]);
    const f32x4 y = ldv4(&be[s0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = s0 + i <= r ? x[i] * y[i] : 0.f;  // (no later token's NaN in an earlier row)
    float* dst = A.X + (row + (int64_t)r * H) * 64 + s0;
    *reinterpret_cast<f32x4*>(dst) = x;
    *reinterpret_cast<f32x4*>(dst + A.mat) = ldv4(&Ps[r * LDL + s0]);
  }
  if (tid < nt) {
    const double bc = bs[C - 1];
    const float e = expf((float)bs[tid]);
    A.aux[row + (int64_t)tid * H] = f32x4{e * nk[tid], e * nq[tid], expf((float)(bc - bs[tid])) * nk[tid], expf((float)bc)};
  }
}

// Workgroup (head, block of 64 value columns, sequence), the portion's chunks in order; layouts as in delta_chunk: a register of an
// accumulator tile is the second operand of a 16x16x4 instruction over its rows 4 g + i, and the first operand's matching numbers are four
// neighbours of a row in LDS. Blocks of 16 tokens past the portion's end are skipped.
// Bound by the chain of a chunk's products, reads and barriers: of 14.3 us a chunk the fp32 matrix instructions took 6.2, now of 12.0 (8 x 1024
// tokens, 16 heads of 128 x 128, 229 -> 192 us). NH = 2 (keys of more than 32): two waves a SIMD, 8 a workgroup; two share 16 columns, each with half of the state's rows (its part of K S and Q S over those; its rows of the update) and
// two of the four blocks of tokens (0 and 3, 1 and 2: five products each with X and with P). Parts of sums, u and U change hands through LDS.
// ANEW: every chunk forms its places anew. Kept through the loop they take what registers are left, and at keys of up to 32 and beyond 64 six and nine
// of them in scratch. A long chain of chunks is still the faster one with them kept (us, kept and anew: one portion of 4096, 8 heads, keys of 32 384
// and 412, of 128 681 and 707; 16 of 256, 32 x 128 82.8 and 83.4), portions of one or two are not (64 of 64, 16 heads of 32 x 128 97 and 90, of 128
// x 128 172 and 166; 100 of 40, 32 x 256 178 and 165; 64 of 24, 128 x 128 125 and 120); keys of 64, with none in scratch, 1 % slower anew.
template <int KT, int NH, bool ANEW>
__global__ __launch_bounds__(256 * NH, KT <= 2 ? 2 : 1) void delta_chunk32_kernel(DeltaChunk32Args A) {
  constexpr int C = 64, DKP = 16 * KT, LDK = DKP + 4, LDP = 64 + 4, KO = KT / NH, TH = 256 * NH;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* Qs = reinterpret_cast<float*>(smem);
  float* Ks = Qs + C * LDK;
  float* Ms = Ks + C * LDK;                                // [2][64][LDP]: X, P
  f32x4* ax = reinterpret_cast<f32x4*>(Ms + 2 * C * LDP);  // [64]
  f32x4* ex = ax + C;                                      // [8 waves][2][2][64 lanes] parts of K S and Q S (NH = 2)
  f32x4* ux = ex + 8 * 4 * 64;                             // [4][4][64] u
  f32x4* uX = ex;                                          // [4][4][64] U: the parts are read by then
  const int h = blockIdx.x, b = gridDim.z - 1 - blockIdx.z;
  const int dim = A.dim, vdim = A.vdim, H = A.H, gq = h / (H / A.G);
  const int t0 = A.cu[b], qlen = A.cu[b + 1] - t0, slot = A.sslots[b], ctx = A.ctx[b];
  if (qlen <= 0) return;
  int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3, hf = wave >> 2;
  const int col = blockIdx.y * 64 + 16 * w + li, colc = min(col, vdim - 1);
  float* outp = A.out + (int64_t)t0 * H * vdim + (int64_t)h * vdim + col;
  if (slot < 0 || ctx <= 0) {
    if (g == 0 && col < vdim && hf == 0)
      for (int j = 0; j < qlen; ++j) outp[(int64_t)j * H * vdim] = 0.f;
    return;
  }
  const bool cont = ctx > qlen;  // continues an earlier portion
  constexpr int NO = 4 / NH;  // blocks of this wave: 0 and 3, 1 and 2
  auto own = [&](int rt) { return NH == 1 || hf == ((rt ^ (rt >> 1)) & 1); };
  auto block = [&](int n) { return NH == 1 ? n : n ? 3 - hf : hf; };
  const int k0w = NH == 1 ? 0 : 16 * KO * hf;                                   // first of this wave's rows of the state
  f32x4 S[KO];
  float* sp = A.S + (((int64_t)slot * H + h) * dim) * (int64_t)vdim;
  load_state(S, cont, sp, k0w + 4 * g, dim, vdim, col);
  constexpr int CHK = DKP / 4, NK = C * CHK / TH, NM = 8 / NH;
  f32x4 rq[NK], rk[NK], rm[NM];
  f32x4 rv[NO];
  f32x4 ra = {0.f, 0.f, 0.f, 0.f};
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  // (the portion's last row again and again past its end, a row's first piece past its last; what is not there becomes zero where it is
  // staged: a zero put in here waits for the load)
  auto fetch = [&](int j0) {
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + TH * j, r = c / CHK, d = (c % CHK) * 4;
      const int64_t tt = t0 + min(j0 + r, qlen - 1), at = (int64_t)gq * dim + (d < dim ? d : 0);
      rq[j] = ldv4(A.q + tt * A.ldq + at);
      rk[j] = ldv4(A.k + tt * A.ldk + at);
    }
#pragma unroll
    for (int j = 0; j < NM; ++j) {
      const int c = tid + TH * j, r = (c >> 4) & 63, s0 = (c & 15) * 4;
      rm[j] = ldv4(A.X + (c >> 10) * A.mat + ((int64_t)(t0 + min(j0 + r, qlen - 1)) * H + h) * 64 + s0);
    }
#pragma unroll
    for (int n = 0; n < NO; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i)  // this lane's column of the blocks' tokens
        rv[n][i] = A.v[(int64_t)(t0 + min(j0 + 16 * block(n) + 4 * g + i, qlen - 1)) * A.ldv + (int64_t)h * vdim + colc];
    ra = A.aux[(int64_t)(t0 + min(j0 + lane, qlen - 1)) * H + h];
  };
  fetch(0);
  // A chunk; ALL: of 64 tokens, without a branch between its blocks, across which no read is moved ahead
  auto chunk = [&](int j0, auto all_c) {
    constexpr bool ALL = decltype(all_c)::value;
    const int nt = ALL ? C : min(C, qlen - j0), nb = ALL ? 4 : (nt + 15) >> 4;
    if constexpr (ANEW) {
      tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      lane = tid & 63, li = lane & 15, g = lane >> 4;
    }
    __syncthreads();  // the previous chunk's readers are done
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + TH * j, r = c / CHK, d = (c % CHK) * 4;
      const bool in = (ALL || r < nt) && d < dim;
      *reinterpret_cast<f32x4*>(&Qs[r * LDK + d]) = in ? rq[j] : zero4;
      *reinterpret_cast<f32x4*>(&Ks[r * LDK + d]) = in ? rk[j] : zero4;
    }
#pragma unroll
    for (int j = 0; j < NM; ++j) {
      const int c = tid + TH * j, r = (c >> 4) & 63;
      *reinterpret_cast<f32x4*>(&Ms[(c >> 10) * C * LDP + r * LDP + (c & 15) * 4]) = ALL || r < nt ? rm[j] : zero4;
    }
    if (wave == 0) ax[lane] = ra;
    f32x4 v[NO], o[NO], ks[NO];  // of this wave's blocks: v first V, then V - e^b K S_0, then U
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      o[n] = ks[n] = zero4;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[n][i] = ALL || 16 * block(n) + 4 * g + i < nt ? rv[n][i] : 0.f;
    }
    __syncthreads();
    if (j0 + C < qlen) fetch(j0 + C);
    const float a_all = ax[0][3];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      if (rt >= nb) continue;
      f32x4 xk[KO], xq[KO];  // (all of a block's reads before its products)
#pragma unroll
      for (int kt = 0; kt < KO; ++kt) {
        xk[kt] = ldv4(&Ks[(16 * rt + li) * LDK + k0w + 4 * g + 16 * kt]);
        xq[kt] = ldv4(&Qs[(16 * rt + li) * LDK + k0w + 4 * g + 16 * kt]);
      }
      __builtin_amdgcn_sched_barrier(0);
      const f32x4 kp = dot32s<KO>(xk, S), qp = dot32s<KO>(xq, S);
      if constexpr (NH == 1) {
        ks[rt] = kp, o[rt] = qp;
      } else {  // one of two blocks is the other wave's
        const int n = rt >> 1;
        const bool mine = own(rt);
        f32x4* const at = ex + ((wave * 2 + n) * 2) * 64 + lane;
        if (rt & 1) {
          const f32x4 kx = mine ? ks[n] : kp, qx = mine ? o[n] : qp;
          at[0] = kx, at[64] = qx;
          ks[n] = mine ? kp : ks[n], o[n] = mine ? qp : o[n];
        } else {
          ks[n] = kp, o[n] = qp;
        }
      }
    }
    if (NH == 2 && (nb & 1)) {  // (its second half was not taken)
      const int n = nb >> 1;
      if (!own(nb - 1)) ex[((wave * 2 + n) * 2) * 64 + lane] = ks[n], ex[((wave * 2 + n) * 2 + 1) * 64 + lane] = o[n];
    }
    if (NH == 2) __syncthreads();
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      const int rt = block(n);
      if (rt >= nb) {
        ks[n] = o[n] = zero4;
        continue;
      }
      if (NH == 2) {
        ks[n] += ex[(((wave ^ 4) * 2 + n) * 2) * 64 + lane];
        o[n] += ex[(((wave ^ 4) * 2 + n) * 2 + 1) * 64 + lane];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 x = ax[16 * rt + 4 * g + i];
        v[n][i] = fmaf(-x[0], ks[n][i], v[n][i]);
        o[n][i] *= x[1];
      }
    }
    f32x4 u[4];  // all blocks
    auto gather = [&](f32x4* at) {
      if constexpr (NH == 2) {
#pragma unroll
        for (int n = 0; n < NO; ++n) at[(w * 4 + block(n)) * 64 + lane] = v[n];
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) u[rt] = at[(w * 4 + rt) * 64 + lane];
      } else {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) u[rt] = v[rt];
      }
      const int bad = contain(u, g);
      if (__builtin_expect(__any(bad < C), 0)) {
#pragma unroll
        for (int n = 0; n < NO; ++n) from_bad(o[n], bad, block(n), g);
      }
      return bad;
    };
    // y += M u of this wave's blocks, M lower triangular. Two blocks (h = 0: 0 and 3, 1: 1 and 2): the first block's first product, the second's
    // first three, and one that is either's.
    auto product = [&](const f32x4& x, const f32x4& y, f32x4 sum) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], sum, 0, 0, 0);
      return sum;
    };
    auto lower = [&](const float* M, f32x4 (&y)[NO]) {
      auto part = [&](int rt, int m) { return ldv4(M + (16 * rt + li) * LDP + 16 * m + 4 * g); };
      if constexpr (NH == 2) {
        const f32x4 x0 = part(hf, 0), x1 = part(3 - hf, 0), x2 = part(3 - hf, 1), x3 = part(3 - hf, 2), x4 = part(hf ? 1 : 3, hf ? 1 : 3);
        const f32x4 ue = hf ? u[1] : u[3];
        const f32x4 a = product(x0, u[0], zero4), f = product(x3, u[2], product(x2, u[1], product(x1, u[0], zero4)));
        const f32x4 e = product(x4, ue, hf ? a : f);
        y[0] += hf ? e : a;
        y[1] += hf ? f : e;
      } else {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          if (rt >= nb) continue;
          f32x4 sum = zero4;
#pragma unroll
          for (int m = 0; m <= rt; ++m) sum = product(part(rt, m), u[m], sum);
          y[rt] += sum;
        }
      }
    };
    // U = X u, O += P U
    int bad = gather(ux);
#pragma unroll
    for (int n = 0; n < NO; ++n) v[n] = zero4;
    lower(Ms, v);
    bad = min(bad, gather(uX));
    lower(Ms + C * LDP, o);
    // the state: e^(b_C) S_0 + K^T (w U)
    const float keep = bad < C ? __uint_as_float(0x7fc00000u) : a_all;
#pragma unroll
    for (int kt = 0; kt < KO; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[kt][i] *= keep;
    f32x4 xs[KO], xw;
    auto columns = [&](int m) {
#pragma unroll
      for (int kt = 0; kt < KO; ++kt) {
        const float* p = &Ks[(16 * m + 4 * g) * LDK + k0w + 16 * kt + li];
        xs[kt] = f32x4{p[0], p[LDK], p[2 * LDK], p[3 * LDK]};
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) xw[i] = ax[16 * m + 4 * g + i][2];
    };
    columns(0);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      if (m >= nb) continue;
      f32x4 x[KO];
#pragma unroll
      for (int kt = 0; kt < KO; ++kt) x[kt] = xs[kt];
      const f32x4 wu = u[m] * xw;
      if (m < 3) columns(m + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int kt = 0; kt < KO; ++kt) S[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[kt][i], wu[i], S[kt], 0, 0, 0);
    }
    if (col < vdim) {
#pragma unroll
      for (int n = 0; n < NO; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * block(n) + 4 * g + i;
          if (ALL || t < nt) outp[(int64_t)(j0 + t) * H * vdim] = o[n][i];
        }
    }
  };
  int j0 = 0;
  if constexpr (NH == 2)
    for (; j0 + C <= qlen; j0 += C) chunk(j0, std::true_type{});
  for (; j0 < qlen; j0 += C) chunk(j0, std::false_type{});
  int r0 = k0w + 4 * g;
  asm volatile("" : "+v"(r0));  // (the rows anew: which of them the state has would be kept in spilled registers through the loop)
  if (col < vdim) {
#pragma unroll
    for (int kt = 0; kt < KO; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + 16 * kt + i;
        if (r < dim) sp[(int64_t)r * vdim + col] = S[kt][i];
      }
  }
}

// (above 128 the chunk's rows and matrices do not fit in LDS)
bool delta_chunk32_ok(int dim, int vdim) { return dim % 4 == 0 && dim >= 4 && dim <= 128 && vdim >= 1; }

// q, k, v fp32, a and b in storage type dp; max_qlen: rows of the longest portion; work: fp32 [2][T, H, 64]; aux: fp32 [T, H, 4]
void launch_delta_chunk32(const void* q, const void* k, const void* v, int64_t ldq, int64_t ldk, int64_t ldv, const void* a,
                          const void* b, int64_t ldab, const void* A_log, const void* dt_bias, void* S, const void* cu,
                          const void* ctx, const void* sslots, void* out, void* work, void* aux, int T_, int B, int max_qlen,
                          int H, int G, int dim, int vdim, int dp, hipStream_t st) {
  if (B == 0 || max_qlen <= 0) return;
  if (!delta_chunk32_ok(dim, vdim) || B > 65535 || H > 65535 || G < 1 || H % G) throw std::runtime_error("delta_chunk32: shape");
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)work | (uintptr_t)aux) & 15 || (ldq | ldk) & 3)
    throw std::runtime_error("delta_chunk32: rows must be 16-byte aligned");
  DeltaChunk32Args A{(const float*)q, (const float*)k, (const float*)v, ldq, ldk, ldv, a, b, ldab, (const float*)A_log,
                     (const float*)dt_bias, (float*)S, (const int*)cu, (const int*)ctx, (const int*)sslots, (float*)out,
                     (float*)work, (int64_t)T_ * H * 64, (f32x4*)aux, H, G, dim, vdim};
  dim3 g1((max_qlen + 63) / 64, H, B), g2(H, (vdim + 63) / 64, B);
  auto lds1 = [](int kt) { return (size_t)prep32_k_bytes(kt) + (size_t)4 * (64 * 68 + 3 * 64) + 8 * 64; };
  // (two halves: parts of sums, u and U besides)
  auto lds2 = [](int kt, int nh) { return (size_t)4 * (2 * 64 * (16 * kt + 4) + 2 * 64 * 68) + (size_t)16 * 64 + (nh == 2 ? 16 * 64 * 48 : 0); };
#define LAUNCH_DC32(KT_, NH_)                                                                                         \
  do {                                                                                                                \
    static bool once = [] {                                                                                           \
      for (const void* f : {(const void*)delta_prep32_kernel<KT_, bf16_t>, (const void*)delta_prep32_kernel<KT_, float>,\
                            (const void*)delta_chunk32_kernel<KT_, NH_, false>, (const void*)delta_chunk32_kernel<KT_, NH_, KT_ != 4>}) \
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                         \
      return true;                                                                                                    \
    }();                                                                                                              \
    (void)once;                                                                                                       \
    DISPATCH_T(dp, TP, (delta_prep32_kernel<KT_, TP><<<g1, 256, lds1(KT_), st>>>(A)));                                \
    if (max_qlen <= 128) delta_chunk32_kernel<KT_, NH_, KT_ != 4><<<g2, 256 * NH_, lds2(KT_, NH_), st>>>(A);          \
    else delta_chunk32_kernel<KT_, NH_, false><<<g2, 256 * NH_, lds2(KT_, NH_), st>>>(A);                             \
  } while (0)
  if (dim <= 32) LAUNCH_DC32(2, 1);
  else if (dim <= 64) LAUNCH_DC32(4, 2);
  else LAUNCH_DC32(8, 2);
#undef LAUNCH_DC32
  HIP_CHECK_LAUNCH();
}
