// The linear matrix recurrences - constant decay (decay) and the state-space scan (ssd) - in the two forms that carry a serving
// step, beside the token-by-token walk of recurrent.hip. Per head, with g = decay[head] and e = 1, or with
// e = softplus(dt + dt_bias[head]) and g = exp(-exp(A_log[head]) e):
//   S <- g S + e k v^T,  o = S^T q (+ D[head] v)
//
//   linear_step:   steps of single rows. One workgroup per (sequence, head): one pass over the state in 16-byte accesses (columns
//                  over lanes, state rows over groups of threads), all of a thread's rows in flight at once.
//   linear_chunk:  portions of bf16 rows on the matrix cores, 64 tokens at a time. With F_t the sum of log g from the chunk's
//                  start to t and S_0 the state before it,
//                    o_t = e^(F_t) S_0^T q_t + sum_{s <= t} e^(F_t - F_s) e_s (q_t . k_s) v_s
//                    S_C = e^(F_C) S_0 + sum_s e^(F_C - F_s) e_s k_s v_s^T
//                  four matrix products per chunk with 32-bit operands, sums and state, as in the walk; F is summed in 64 bits, so
//                  that a difference of two large sums is as good as the factor it stands for. decay, whose rows pass through an
//                  activation first, runs on the fp32 matrix instructions. ssd's q and k are exact in bf16: a product with them
//                  takes the 32-bit factor as three bf16 numbers that add up to it exactly and runs on the bf16 instructions,
//                  at three sixteenths of the fp32 ones' cost.
#include <type_traits>

#include "anytype.h"
#include "chunk_rows.h"

struct LinearArgs {
  const void* q;  // [T, ldq]: head group's query at q + (h / rep) * dim
  const void* k;
  const void* v;  // head h's values at v + h * vdim
  int64_t ldq, ldk, ldv;
  const void* dt;  // ssd: [T, lddt], one step size per head before bias and softplus
  int64_t lddt;
  const float* decay;    // decay: [H]; ssd: A_log [H]
  const float* dt_bias;  // ssd: [H]
  const float* skip;     // ssd: D [H]
  float* S;              // [slots, H, dim, vdim]
  const int* cu;
  const int* ctx;
  const int* sslots;
  float* out;  // [T, H * vdim]
  int H, G, dim, vdim, silu;  // silu: q, k and v pass through it first
};

template <typename T>
__device__ __forceinline__ float lin_silu(float v) {  // bf16 rows: the fast exponential, as in the walk
  return v / (1.0f + (sizeof(T) == 2 ? __expf(-v) : expf(-v)));
}
__device__ __forceinline__ float lin_softplus(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// ------------------------------------------------------------------------------------------------ single rows
// Bound by the state's bytes, read and written once. 64 sequences: ssd, 64 heads 128 x 64, 128 -> 42 us (268 MB, 6.3 TB/s);
// decay, 16 heads 128 x 128, 44 -> 22 us (134 MB). The walk's columns, split over 4 lanes, touch 64-byte runs and keep 32 loads
// of 4 bytes in flight per lane; here a thread has up to 32 of 16 bytes.
// U: state rows per thread
template <typename T, int MODE, int U>
__global__ __launch_bounds__(256) void linear_step_kernel(LinearArgs A) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int dim = A.dim, vdim = A.vdim, H = A.H, gq = h / (H / A.G);
  const int t = A.cu[b], slot = A.sslots[b], pos = A.ctx[b] - 1;
  float* outp = A.out + ((int64_t)t * H + h) * vdim;
  if (slot < 0 || pos < 0) {
    for (int c = tid; c < vdim; c += 256) outp[c] = 0.f;
    return;
  }
  float* qs = sm;                        // [dim]
  float* ks = qs + dim;                  // [dim], times e
  float* part = sm + ((2 * dim + 3) & ~3);  // [row groups][vdim]
  // thread (rg, cg): columns 4 cg .. 4 cg + 3 of the state rows rg, rg + RG, ...
  const int ncg = vdim >> 2, RG = 256 / ncg, cg = tid % ncg, rg = tid / ncg;
  float* sp = A.S + (((int64_t)slot * H + h) * dim) * (int64_t)vdim + 4 * cg;
  f32x4 s[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = rg + u * RG;
    s[u] = (pos > 0 && rg < RG && r < dim) ? *reinterpret_cast<const f32x4*>(sp + (int64_t)r * vdim) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float a, e = 1.0f;
  if (MODE == 2) {
    e = lin_softplus(El<T>::ld((const T*)A.dt + (int64_t)t * A.lddt + h) + A.dt_bias[h]);
    a = expf(-expf(A.decay[h]) * e);
  } else {
    a = A.decay[h];
  }
  const T* qr = (const T*)A.q + (int64_t)t * A.ldq + (int64_t)gq * dim;
  const T* kr = (const T*)A.k + (int64_t)t * A.ldk + (int64_t)gq * dim;
  for (int d = tid; d < dim; d += 256) {
    const float qd = El<T>::ld(qr + d), kd = El<T>::ld(kr + d);
    qs[d] = A.silu ? lin_silu<T>(qd) : qd;
    ks[d] = e * (A.silu ? lin_silu<T>(kd) : kd);
  }
  __syncthreads();
  const T* vr = (const T*)A.v + (int64_t)t * A.ldv + (int64_t)h * vdim;
  if (rg < RG) {
    f32x4 v4, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = El<T>::ld(vr + 4 * cg + i);
      v4[i] = A.silu ? lin_silu<T>(x) : x;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = rg + u * RG;
      if (r < dim) {
        const float kd = ks[r], qd = qs[r];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[u][i] = fmaf(a, s[u][i], kd * v4[i]);
          o[i] = fmaf(s[u][i], qd, o[i]);
        }
        *reinterpret_cast<f32x4*>(sp + (int64_t)r * vdim) = s[u];
      }
    }
    *reinterpret_cast<f32x4*>(part + (int64_t)rg * vdim + 4 * cg) = o;
  }
  __syncthreads();
  for (int c = tid; c < vdim; c += 256) {
    float o = 0.f;
    for (int r = 0; r < RG; ++r) o += part[r * vdim + c];
    if (MODE == 2 && A.skip) o = fmaf(A.skip[h], El<T>::ld(vr + c), o);
    outp[c] = o;
  }
}

static int linear_step_rows(int dim, int vdim) {  // state rows per thread (0: the shape does not fit)
  if (vdim % 4 || vdim < 4 || vdim > 1024 || dim < 1 || dim > 512) return 0;  // (512: the walk's largest; 8 KB of LDS here)
  const int RG = 256 / (vdim / 4), U = (dim + RG - 1) / RG;
  return U <= 32 ? U : 0;
}
bool linear_step_ok(int dim, int vdim) { return linear_step_rows(dim, vdim) > 0; }

template <typename T, int MODE>
static void linear_step_t(const LinearArgs& A, int B, hipStream_t st) {
  const int U = linear_step_rows(A.dim, A.vdim), RG = 256 / (A.vdim / 4);
  const size_t lds = ((size_t)2 * A.dim + 4 + (size_t)RG * A.vdim) * 4;
  dim3 g(A.H, B);
  if (U <= 8) linear_step_kernel<T, MODE, 8><<<g, 256, lds, st>>>(A);
  else if (U <= 16) linear_step_kernel<T, MODE, 16><<<g, 256, lds, st>>>(A);
  else linear_step_kernel<T, MODE, 32><<<g, 256, lds, st>>>(A);
}

static LinearArgs linear_args(int mode, const void* q, const void* k, const void* v, int64_t ldq, int64_t ldk, int64_t ldv,
                              const void* dt, int64_t lddt, const void* decay, const void* dt_bias, const void* skip, void* S,
                              const void* cu, const void* ctx, const void* sslots, void* out, int H, int G, int dim, int vdim,
                              int silu) {
  if (mode != 0 && mode != 2) throw std::runtime_error("linear scan: mode");
  if (G < 1 || H % G) throw std::runtime_error("linear scan: heads must be a multiple of the key heads");
  return LinearArgs{q, k, v, ldq, ldk, ldv, dt, lddt, (const float*)decay, (const float*)dt_bias, (const float*)skip, (float*)S,
                    (const int*)cu, (const int*)ctx, (const int*)sslots, (float*)out, H, G, dim, vdim, silu};
}

// B sequences of one row each; q, k, v and dt in one storage type
void launch_linear_step(int mode, const void* q, const void* k, const void* v, int64_t ldq, int64_t ldk, int64_t ldv,
                        const void* dt, int64_t lddt, const void* decay, const void* dt_bias, const void* skip, void* S,
                        const void* cu, const void* ctx, const void* sslots, void* out, int B, int H, int G, int dim, int vdim,
                        int silu, int dtype, hipStream_t st) {
  if (B == 0) return;
  const LinearArgs A = linear_args(mode, q, k, v, ldq, ldk, ldv, dt, lddt, decay, dt_bias, skip, S, cu, ctx, sslots, out, H, G,
                                   dim, vdim, silu);
  if (!linear_step_ok(dim, vdim) || B > 65535) throw std::runtime_error("linear_step: shape");
  if ((uintptr_t)S & 15) throw std::runtime_error("linear_step: the state must be 16-byte aligned");
  DISPATCH_T(dtype, T, {
    if (mode == 0) linear_step_t<T, 0>(A, B, st);
    else linear_step_t<T, 2>(A, B, st);
  });
  HIP_CHECK_LAUNCH();
}

// ------------------------------------------------------------------------------------------------ portions
struct Split3 {  // eight numbers, each the sum of three
  s16x8 h, m, l;
};
__device__ __forceinline__ f32x4 lin_mfma3(const s16x8& a, const Split3& b, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.l, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.m, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.h, c, 0, 0, 0);
}
__device__ __forceinline__ s16x8 lin_cat(const s16x4& a, const s16x4& b) {
  return s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// A value that is infinite or NaN makes, by zeros of the scores times it, the tokens before it in its block of 16 NaN as well, which a walk
// token by token does not. Their results once more, by such a walk from the portion's start: a wave for its 16 columns from col0 on, those
// in `lanes` (a column has four), which the state tells: it has taken the value. Written for the rare case; in the chunks' loop a
// branch for it cost 200 -> 244 us (8 x 1024 tokens, 64 heads 128 x 64).
template <int MODE>
__device__ __forceinline__ void linear_mend(const LinearArgs& A, int h, int b, int col0, uint64_t lanes, int lane) {
  const int t0 = A.cu[b], qlen = A.cu[b + 1] - t0, dim = A.dim, vdim = A.vdim, gq = h / (A.H / A.G);
  const bool cont = A.ctx[b] > qlen;
  const float* sp = A.S + (((int64_t)A.sslots[b] * A.H + h) * dim) * (int64_t)vdim;
  const uint64_t cols = lanes | lanes >> 16 | lanes >> 32 | lanes >> 48;
  for (int c = 0; c < 16; ++c) {
    const int col = col0 + c;
    if (!(cols >> c & 1) || col >= vdim) continue;
    auto value = [&](int t) {
      const float x = bf2f(((const bf16_t*)A.v)[(int64_t)(t0 + t) * A.ldv + (int64_t)h * vdim + col]);
      return MODE == 0 && A.silu ? lin_silu<bf16_t>(x) : x;
    };
    int bad = qlen;
    for (int t = lane; t < qlen; t += 64)
      if (!(fabsf(value(t)) <= FLT_MAX)) bad = min(bad, t);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) bad = min(bad, __shfl_xor(bad, o, 64));
    if (bad % 16 == 0 || bad == qlen) continue;
    float S[4];  // rows lane, lane + 64, ...
#pragma unroll
    for (int i = 0; i < 4; ++i) S[i] = cont && lane + 64 * i < dim ? sp[(int64_t)(lane + 64 * i) * vdim + col] : 0.f;
    for (int t = 0; t < bad; ++t) {
      const int64_t tt = t0 + t;
      float a = A.decay[h], e = 1.f, acc = 0.f;
      if (MODE == 2) {
        e = lin_softplus(bf2f(((const bf16_t*)A.dt)[tt * A.lddt + h]) + A.dt_bias[h]);
        a = expf(-expf(a) * e);
      }
      const float x = value(t);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (lane + 64 * i < dim) {
          const int64_t d = (int64_t)gq * dim + lane + 64 * i;
          const float k = bf2f(((const bf16_t*)A.k)[tt * A.ldk + d]), q = bf2f(((const bf16_t*)A.q)[tt * A.ldq + d]);
          S[i] = fmaf(a, S[i], e * (A.silu ? lin_silu<bf16_t>(k) : k) * x);
          acc = fmaf(S[i], A.silu ? lin_silu<bf16_t>(q) : q, acc);
        }
      acc = warp_sum(acc);
      if (MODE == 2 && A.skip) acc = fmaf(A.skip[h], x, acc);
      if (t >= (bad & ~15) && lane == 0) A.out[(tt * A.H + h) * vdim + col] = acc;
    }
  }
}

// Bound by the chain of chunks: a prompt step of 8 sequences has one (decay) or two (ssd) workgroups per CU, each 16 dependent
// chunks. 8 x 1024 tokens: ssd, 64 heads 128 x 64, 2160 us token by token, 310 us with fp32 instructions throughout, 182 us here
// (no workgroup exchanges anything inside a chunk but the scores); decay, 16 heads 128 x 128, 1230 us with its activation pass,
// 256 us here.
//
// Workgroup (head, block of 64 value columns, sequence), 4 waves, the portion's chunks in order. A wave owns 16 value columns:
// its part of the state lives in registers in the accumulator layout (lane (li, g): column li, rows 16 tile + 4 g + i), and so do
// V and its weighted form over the tokens. Register i of such a tile is, as it stands, the second operand of a 16x16x4
// instruction whose four k are the rows 4 g + i; the first operand's matching numbers are four neighbours of a row in LDS (one
// wide read per four instructions); a 16x16x32 instruction takes the eight rows 4 g + i of two neighbouring tiles likewise. Blocks
// of 16 tokens past the portion's end are skipped. q and k stay bf16 in LDS where they are used as stored, and are held in 32 bits where the
// activation comes first. The next chunk's rows are fetched into registers while this one is computed. KT: 16-row tiles of the
// state (dim padded with zeros).
template <int KT, int MODE>
__global__ __launch_bounds__(256, KT <= 4 || (MODE == 2 && KT <= 8) ? 2 : 1) void linear_chunk_kernel(LinearArgs A) {
  using LT = typename std::conditional<MODE == 2, bf16_t, float>::type;
  constexpr int C = 64, DKP = 16 * KT, LDK = DKP + (MODE == 2 ? 8 : 4), LDP = 64 + 4;
  constexpr int NCH = KT < 4 ? 2 : 4;  // chains an fp32 product over the keys is summed in: shorter ones round less
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  LT* Qs = reinterpret_cast<LT*>(smem);
  LT* Ks = Qs + C * LDK;
  float* Ps = reinterpret_cast<float*>(Ks + C * LDK);  // [64][LDP]
  double* Fs = reinterpret_cast<double*>(Ps + C * LDP);  // [64]
  float* es = reinterpret_cast<float*>(Fs + C);          // [64] e_s
  float* gt = es + C;                                    // [64] e^(F_t)
  float* ws = gt + C;                                    // [64] e^(F_C - F_s) e_s
  const int h = blockIdx.x, b = gridDim.z - 1 - blockIdx.z;
  const int dim = A.dim, vdim = A.vdim, H = A.H, gq = h / (H / A.G);
  const int t0 = A.cu[b], qlen = A.cu[b + 1] - t0, slot = A.sslots[b], ctx = A.ctx[b];
  if (qlen <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, g = lane >> 4;
  const int col = blockIdx.y * 64 + 16 * w + li, colc = min(col, vdim - 1);
  float* outp = A.out + ((int64_t)t0 * H + h) * vdim + col;
  if (slot < 0 || ctx <= 0) {
    if (g == 0 && col < vdim)
      for (int j = 0; j < qlen; ++j) outp[(int64_t)j * H * vdim] = 0.f;
    return;
  }
  const bool cont = ctx > qlen;  // continues an earlier portion
  f32x4 S[KT];
  float* sp = A.S + (((int64_t)slot * H + h) * dim) * (int64_t)vdim;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) S[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // (numbers that are not there are read from the nearest place that is and replaced afterwards, here and in the rows below: behind a
  // condition of its own, or with its zero beside it, every load was waited for before the next)
  if (cont) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[kt][i] = sp[(int64_t)min(16 * kt + 4 * g + i, dim - 1) * vdim + colc];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[kt][i] = 16 * kt + 4 * g + i < dim && col < vdim ? S[kt][i] : 0.f;
  }
  constexpr int CHK = DKP / 8, NK = C * CHK / 256;
  static_assert((C * CHK) % 256 == 0, "whole 16-byte pieces per thread");
  u16x8 rq[NK], rk[NK];
  uint32_t rv[16], rd = 0;  // (words: two numbers to a register wait for both)
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  auto fetch = [&](int j0) {  // the portion's last row again and again past its end, a row's first piece past its last
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 8;
      const int64_t tt = t0 + min(j0 + r, qlen - 1), at = (int64_t)gq * dim + (d < dim ? d : 0);
      rq[j] = *reinterpret_cast<const u16x8*>((const bf16_t*)A.q + tt * A.ldq + at);
      rk[j] = *reinterpret_cast<const u16x8*>((const bf16_t*)A.k + tt * A.ldk + at);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {  // token 16 (j / 4) + 4 g + j % 4 at this lane's column
      const int r = j0 + 16 * (j >> 2) + 4 * g + (j & 3);
      rv[j] = ((const bf16_t*)A.v)[(int64_t)(t0 + min(r, qlen - 1)) * A.ldv + (int64_t)h * vdim + colc];
    }
    if (MODE == 2) rd = ((const bf16_t*)A.dt)[(int64_t)(t0 + min(j0 + lane, qlen - 1)) * A.lddt + h];
  };
  // rows into LDS and V into registers; the choice of the activation is made once for all of them (at each number it cost more than the
  // number, one after the other: decay, 16 heads 128 x 128 of 8 x 1024 tokens, with the places and factors read ahead 369 -> 256 us)
  auto stage_as = [&](int j0, f32x4 (&v)[4], auto silu_c) {
    constexpr bool SILU = decltype(silu_c)::value;
    auto stage = [&](LT* dst, const u16x8& x) {
      if constexpr (MODE == 2) {
        *reinterpret_cast<u16x8*>(dst) = x;
      } else {
        f32x4 lo, hi;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float u = bf2f(x[i]), z = bf2f(x[4 + i]);
          lo[i] = SILU ? lin_silu<bf16_t>(u) : u;
          hi[i] = SILU ? lin_silu<bf16_t>(z) : z;
        }
        *reinterpret_cast<f32x4*>(dst) = lo;
        *reinterpret_cast<f32x4*>(dst + 4) = hi;
      }
    };
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + 256 * j, r = c / CHK, d = (c % CHK) * 8;
      const bool in = j0 + r < qlen && d < dim;
      stage(&Qs[r * LDK + d], in ? rq[j] : zero8);
      stage(&Ks[r * LDK + d], in ? rk[j] : zero8);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float x = j0 + 16 * (j >> 2) + 4 * g + (j & 3) < qlen ? bf2f((bf16_t)rv[j]) : 0.f;
      v[j >> 2][j & 3] = MODE == 0 && SILU ? lin_silu<bf16_t>(x) : x;
    }
  };
  const float dskip = MODE == 2 && A.skip ? A.skip[h] : 0.f;
  const float dec = A.decay[h];
  // the log factor of a token; a factor of zero (or nearly so) becomes one that vanishes over a single token
  const double lg0 = MODE == 0 ? at_least(log((double)fabsf(dec)), -1e4) : 0.0;
  const bool alt = MODE == 0 && dec < 0.f;  // a negative factor: the sign alternates with the distance
  const float ea = MODE == 2 ? expf(dec) : 0.f, dtb = MODE == 2 ? A.dt_bias[h] : 0.f;
  fetch(0);
  // A chunk; ALL: of 64 tokens, without a branch between its blocks
  auto chunk = [&](int j0, auto all_c) {
    constexpr bool ALL = decltype(all_c)::value;
    const int nt = ALL ? C : min(C, qlen - j0);
    // (the places anew: those of all reads below, kept through the loop, leave no room for the next chunk's rows, and a number in scratch is waited
    // for with every load that is on its way: state space, 64 heads of 128 x 64 over 8 x 1024 tokens, 193 -> 159 us; decay, 16 heads of 128 x 128,
    // 243 -> 228)
    int lo = lane;
    asm volatile("" : "+v"(lo));
    const int li = lo & 15, g = lo >> 4;
    __syncthreads();  // the previous chunk's readers are done
    f32x4 v[4];
    if (MODE != 2 && A.silu) stage_as(j0, v, std::true_type{});
    else stage_as(j0, v, std::false_type{});
    if (w == 0) {
      const bool in = lane < nt;
      double F;
      float e = in ? 1.0f : 0.f;
      if (MODE == 2) {
        e = in ? lin_softplus(bf2f((bf16_t)rd) + dtb) : 0.f;
        F = in ? at_least((double)(-ea * e), -1e8) : 0.0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const double x = __shfl_up(F, o, 64);
          if (lane >= o) F += x;
        }
      } else {
        F = lg0 * (double)min(lane + 1, nt);
      }
      const double FC = __shfl(F, 63, 64);
      Fs[lane] = F;
      es[lane] = e;
      float gv = expf((float)F), wv = expf((float)(FC - F)) * e;
      if (alt) {
        if (min(lane + 1, nt) & 1) gv = -gv;
        if ((nt - 1 - lane) & 1) wv = -wv;
      }
      gt[lane] = gv;
      ws[lane] = wv;
    }
    __syncthreads();
    if (j0 + C < qlen) fetch(j0 + C);
    const int nb = ALL ? 4 : (nt + 15) >> 4;  // blocks of tokens
    // weighted scores: wave w owns the tokens 16 w .. 16 w + 15 (rows) and the keys up to them (columns)
    if (w < nb) {
      f32x4 p[4];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) p[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (MODE == 2) {
#pragma unroll
        for (int ks = 0; ks < KT / 2; ++ks) {
          const s16x8 a = *reinterpret_cast<const s16x8*>(&Qs[(16 * w + li) * LDK + 32 * ks + 8 * g]);
#pragma unroll
          for (int ct = 0; ct < 4; ++ct) {
            if (ct > w) continue;
            const s16x8 x = *reinterpret_cast<const s16x8*>(&Ks[(16 * ct + li) * LDK + 32 * ks + 8 * g]);
            p[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, x, p[ct], 0, 0, 0);
          }
        }
      } else {
        f32x4 a[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) a[kt] = ld4(&Qs[(16 * w + li) * LDK + 16 * kt + 4 * g]);
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          if (ct > w) continue;
          f32x4 c[NCH];
#pragma unroll
          for (int n = 0; n < NCH; ++n) c[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kt = 0; kt < KT; kt += NCH) {
            f32x4 x[NCH];
#pragma unroll
            for (int n = 0; n < NCH; ++n) x[n] = ld4(&Ks[(16 * ct + li) * LDK + 16 * (kt + n) + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int n = 0; n < NCH; ++n) c[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[kt + n][i], x[n][i], c[n], 0, 0, 0);
          }
          p[ct] = NCH == 4 ? (c[0] + c[1]) + (c[NCH - 2] + c[NCH - 1]) : c[0] + c[1];
        }
      }
      double Ft[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) Ft[i] = Fs[16 * w + 4 * g + i];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        if (ct > w) continue;
        const int s = 16 * ct + li;
        const double Fv = Fs[s];
        const float ev = es[s];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * w + 4 * g + i;
          const float f = expf((float)(Ft[i] - Fv)) * ev, z = p[ct][i] * (alt && ((t - s) & 1) ? -f : f);
          Ps[t * LDP + s] = s <= t ? z : 0.f;
        }
      }
    }
    // Q S for this wave's columns while the other waves finish their scores
    f32x4 o[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) o[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (MODE == 2) {
#pragma unroll
      for (int ks = 0; ks < KT / 2; ++ks) {
        Split3 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) split3(S[2 * ks + (j >> 2)][j & 3], j, x.h, x.m, x.l);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          if (rt >= nb) continue;
          const bf16_t* p = &Qs[(16 * rt + li) * LDK + 32 * ks + 4 * g];
          o[rt] = lin_mfma3(lin_cat(*reinterpret_cast<const s16x4*>(p), *reinterpret_cast<const s16x4*>(p + 16)), x, o[rt]);
        }
      }
    } else {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        if (rt >= nb) continue;
        f32x4 c[NCH];
#pragma unroll
        for (int n = 0; n < NCH; ++n) c[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < KT; kt += NCH) {
          f32x4 x[NCH];
#pragma unroll
          for (int n = 0; n < NCH; ++n) x[n] = ld4(&Qs[(16 * rt + li) * LDK + 16 * (kt + n) + 4 * g]);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < NCH; ++n) c[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[n][i], S[kt + n][i], c[n], 0, 0, 0);
        }
        o[rt] = NCH == 4 ? (c[0] + c[1]) + (c[NCH - 2] + c[NCH - 1]) : c[0] + c[1];
      }
    }
    const float gC = gt[C - 1];
    f32x4 vw[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const f32x4 g4 = ld4(&gt[16 * rt + 4 * g]), w4 = ld4(&ws[16 * rt + 4 * g]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o[rt][i] *= g4[i];
        vw[rt][i] = v[rt][i] * w4[i];
      }
    }
    // the state: e^(F_C) S_0 + K^T (w V)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) S[kt][i] *= gC;
    }
    if constexpr (MODE == 2) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        if (2 * ks >= nb) continue;
        Split3 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) split3(vw[2 * ks + (j >> 2)][j & 3], j, x.h, x.m, x.l);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          const bf16_t* p = &Ks[(32 * ks + 4 * g + (li >> 2)) * LDK + 16 * kt + 4 * (li & 3)];
          const s16x4 y0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(p));
          const s16x4 y1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(p + 16 * LDK));
          S[kt] = lin_mfma3(lin_cat(y0, y1), x, S[kt]);
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (m >= nb) continue;
#pragma unroll
        for (int k0 = 0; k0 < KT; k0 += 4) {
          f32x4 a[4];
#pragma unroll
          for (int kt = 0; kt < 4; ++kt)
            if (k0 + kt < KT) {
              const float* p = &Ks[(16 * m + 4 * g) * LDK + 16 * (k0 + kt) + li];
              a[kt] = f32x4{p[0], p[LDK], p[2 * LDK], p[3 * LDK]};
            }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
              if (k0 + kt < KT) S[k0 + kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[kt][i], vw[m][i], S[k0 + kt], 0, 0, 0);
        }
      }
    }
    __syncthreads();  // every wave's weighted scores are in LDS
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      if (rt >= nb) continue;
      f32x4 in = {0.f, 0.f, 0.f, 0.f};  // the chunk's own part, summed apart from the state's
#pragma unroll
      for (int m = 0; m <= rt; ++m) {
        const f32x4 a = ld4(&Ps[(16 * rt + li) * LDP + 16 * m + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) in = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], v[m][i], in, 0, 0, 0);
      }
      o[rt] += in;
    }
    if (col < vdim) {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * rt + 4 * g + i;
          if (ALL || t < nt) outp[(int64_t)(j0 + t) * H * vdim] = MODE == 2 ? fmaf(dskip, v[rt][i], o[rt][i]) : o[rt][i];
        }
    }
  };
  int j0 = 0;
  for (; j0 + C <= qlen; j0 += C) chunk(j0, std::true_type{});
  if (j0 < qlen) chunk(j0, std::false_type{});
  float z = 0.f;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) z = fmaf(S[kt][i], 0.f, z);
  if (__builtin_expect(__any(z != z), 0)) {
    linear_mend<MODE>(A, h, b, blockIdx.y * 64 + 16 * w, __ballot(z != z), lane);
    // (its loads and stores end here: left open, each store of the state below waits for the one before it, on the usual path too)
    __builtin_amdgcn_s_waitcnt(0x0070);
  }
  int r0 = 4 * g;
  asm volatile("" : "+v"(r0));  // (the rows anew: those of the state's loads, kept in scratch through the loop, cost a wait for each store)
  if (col < vdim) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + 16 * kt + i;
        if (r < dim) sp[(int64_t)r * vdim + col] = S[kt][i];
      }
  }
}

bool linear_chunk_ok(int dim, int vdim) { return dim % 8 == 0 && dim >= 8 && dim <= 256 && vdim >= 1; }

// portions of bf16 rows (q, k, v and dt)
void launch_linear_chunk(int mode, const void* q, const void* k, const void* v, int64_t ldq, int64_t ldk, int64_t ldv,
                         const void* dt, int64_t lddt, const void* decay, const void* dt_bias, const void* skip, void* S,
                         const void* cu, const void* ctx, const void* sslots, void* out, int B, int H, int G, int dim, int vdim,
                         int silu, hipStream_t st) {
  if (B == 0) return;
  const LinearArgs A = linear_args(mode, q, k, v, ldq, ldk, ldv, dt, lddt, decay, dt_bias, skip, S, cu, ctx, sslots, out, H, G,
                                   dim, vdim, silu);
  if (!linear_chunk_ok(dim, vdim) || B > 65535 || (vdim + 63) / 64 > 65535 || (mode == 2 && silu))
    throw std::runtime_error("linear_chunk: shape");
  if (((uintptr_t)q | (uintptr_t)k) & 15 || (ldq | ldk) & 7) throw std::runtime_error("linear_chunk: rows must be 16-byte aligned");
  dim3 g(H, (vdim + 63) / 64, B);
  auto lds = [&](int kt) {
    return (size_t)2 * 64 * (mode == 2 ? 2 * (16 * kt + 8) : 4 * (16 * kt + 4)) + (size_t)64 * 68 * 4 + 64 * 8 + 3 * 64 * 4;
  };
#define LAUNCH_LC(KT_, MODE_)                                                                                        \
  do {                                                                                                               \
    static bool once = [] {                                                                                          \
      (void)hipFuncSetAttribute((const void*)linear_chunk_kernel<KT_, MODE_>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                160 * 1024);                                                                         \
      return true;                                                                                                   \
    }();                                                                                                             \
    (void)once;                                                                                                      \
    linear_chunk_kernel<KT_, MODE_><<<g, 256, lds(KT_), st>>>(A);                                                    \
  } while (0)
#define LAUNCH_LCM(KT_)              \
  do {                               \
    if (mode == 2) LAUNCH_LC(KT_, 2); \
    else LAUNCH_LC(KT_, 0);          \
  } while (0)
  if (dim <= 32) LAUNCH_LCM(2);
  else if (dim <= 64) LAUNCH_LCM(4);
  else if (dim <= 128) LAUNCH_LCM(8);
  else LAUNCH_LCM(16);
#undef LAUNCH_LCM
#undef LAUNCH_LC
  HIP_CHECK_LAUNCH();
}
