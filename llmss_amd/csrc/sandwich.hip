// Blocks normed on both sides of a sublayer, over the fp32 residual stream x [T, W]:
//
//   sandwich_add_norm:  x += rms_norm(y * sigmoid(r + rb)) * wpost      y the sublayer's result, r its gate logits
//                       x += add                                        (optional fp32 rows, or one row for all)
//                       h  = rms_norm(x) * wnext                        (optional, in the storage type)
//   token_side_add:     e = table[id, col0 : col0 + d]; g = gelu_tanh(Wg x) * e; y = Wp g;
//                       x += rms_norm(y) * wn, then the same optional `add` and `h`
//
// A norm may be taken in `groups` equal consecutive parts of the row, each divided by its own root mean square
// (groups = 1: the whole row); both norms of a launch take the same number of parts.
//
// so a sublayer's closing op also forms the next reader's input, as add_norm does for the uniform families. y is
// either a dense row in the storage type, or the still uncombined output of a mixture-of-experts layer (moe.hip):
// y[t] = sum_j (wts ? wts[t, j] : 1) * ey[place[t * top + j]] (+ shared[t]), j ascending, then the shared expert.
// A pair whose place is negative chose an identity expert: its output is ident[t], the sublayer's own input row. Or y
// is the result of two mixers side by side, y = 1/2 (rms_norm(y) * wl + rms_norm(y2) * wr), both norms over the whole row,
// or (no wl, wr) y = cl * y + cr * y2. The shared expert's row may carry a factor per token, sw[t].
// Norm weights, biases and layer scales are fp32. One workgroup per row; the gated row lives in LDS between the
// pass that sums its squares and the pass that adds it, and the updated x between that pass and the norm.
#include "anytype.h"
#include "route.h"

struct SandwichArgs {
  float* x;
  const void* y;
  int64_t ldy;
  const float* ey;
  const int* place;
  const float* wts;
  int top;
  const void* shared_;
  int64_t lds_;
  const void* r;
  int64_t ldr;
  const float* rb;
  const float* wpost;
  const float* add;
  const float* wnext;
  void* h;
  int64_t ldh;
  float eps;
  int W;
  int groups;
  const void* ident;  // [T, W] in the storage type
  int64_t ldi;
  const void* y2;
  int64_t ldy2;
  const float* wl;
  const float* wr;
  float cl, cr;
  int64_t lda;      // row stride of add (0: one row for all)
  const float* sw;  // [T] or null
  int slabs;        // > 0: y is the fp32 slabs [slabs][T][W] of a product whose K was split
};

template <typename T, int V>
__device__ __forceinline__ void ldv(const T* p, float* v) {
  if constexpr (V == 4 && sizeof(T) == 4) {
    const f32x4 q = *reinterpret_cast<const f32x4*>(p);
    v[0] = q[0], v[1] = q[1], v[2] = q[2], v[3] = q[3];
  } else if constexpr (V == 4) {
    const u16x4 q = *reinterpret_cast<const u16x4*>(p);
    v[0] = bf2f(q[0]), v[1] = bf2f(q[1]), v[2] = bf2f(q[2]), v[3] = bf2f(q[3]);
  } else {
    v[0] = El<T>::ld(p);
  }
}
template <typename T, int V>
__device__ __forceinline__ void stv(T* p, const float* v) {
  if constexpr (V == 4 && sizeof(T) == 4) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
  } else if constexpr (V == 4) {
    *reinterpret_cast<u16x4*>(p) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
  } else {
    El<T>::st(p, v[0]);
  }
}

// 1 / root mean square of every part of the row in buf, left behind the row: buf[W + g]. A wave per part.
__device__ __forceinline__ void part_inv(float* buf, const SandwichArgs& p) {
  const int n = p.W / p.groups, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  __syncthreads();
  for (int g = threadIdx.x >> 6; g < p.groups; g += nw) {
    float s = 0.f;
    for (int c = lane; c < n; c += 64) s = fmaf(buf[g * n + c], buf[g * n + c], s);
    s = warp_sum(s);
    if (lane == 0) buf[p.W + g] = 1.0f / sqrtf(s / (float)n + p.eps);
  }
  __syncthreads();
}

// the tail both kernels share: buf holds the updated x row; writes h = rms_norm(x) * wnext
template <typename T, int V>
__device__ __forceinline__ void norm_out(float* buf, float ss, const SandwichArgs& p, int t, float* red) {
  if (!p.wnext) return;
  float inv = 0.f;
  const float* invs = nullptr;
  if (p.groups > 1) {
    part_inv(buf, p);
    invs = buf + p.W;
  } else {
    ss = block_sum(ss, red);
    inv = 1.0f / sqrtf(ss / (float)p.W + p.eps);
  }
  T* hr = (T*)p.h + (int64_t)t * p.ldh;
  for (int c = threadIdx.x * V; c < p.W; c += blockDim.x * V) {
    float w[V], o[V];
    ldv<float, V>(p.wnext + c, w);
#pragma unroll
    for (int i = 0; i < V; ++i) o[i] = buf[c + i] * (invs ? invs[(c + i) / (p.W / p.groups)] : inv) * w[i];
    stv<T, V>(hr + c, o);
  }
}

// SLABS: y is slabs, as the kernel of whole rows below takes them, at any alignment: 33 rows of 1600, two launches with the product (K =
// 3200) that leaves four slabs and a gate of odd columns, 16.0 us, 17.3 with the product finished first. (A choice at run time beside the others
// costs rows without slabs a quarter: 1557 x 4096 15.3 -> 19.8 us.)
template <typename T, int V, bool SLABS = false>
__global__ __launch_bounds__(512) void sandwich_add_norm_kernel(SandwichArgs p) {
  extern __shared__ __attribute__((aligned(16))) float buf[];
  __shared__ float red[32];
  const int t = blockIdx.x, W = p.W;
  float* xr = p.x + (int64_t)t * W;
  const bool has_y = p.y != nullptr || p.ey != nullptr;
  float inv = 0.f;
  if (has_y) {
    const T* yr = p.y ? (const T*)p.y + (int64_t)t * p.ldy : nullptr;
    const T* sr = p.shared_ ? (const T*)p.shared_ + (int64_t)t * p.lds_ : nullptr;
    const T* rr = p.r ? (const T*)p.r + (int64_t)t * p.ldr : nullptr;
    const T* y2r = p.y2 ? (const T*)p.y2 + (int64_t)t * p.ldy2 : nullptr;
    float il = 0.f, ir = 0.f;
    if (y2r && p.wl) {  // two mixers: the root mean square of each row first
      float sl = 0.f, sr2 = 0.f;
      for (int c = threadIdx.x * V; c < W; c += blockDim.x * V) {
        float a[V], b[V];
        ldv<T, V>(yr + c, a);
        ldv<T, V>(y2r + c, b);
#pragma unroll
        for (int i = 0; i < V; ++i) {
          sl = fmaf(a[i], a[i], sl);
          sr2 = fmaf(b[i], b[i], sr2);
        }
      }
      const f32x2 s2 = block_sum2(sl, sr2, red);
      il = 0.5f / sqrtf(s2[0] / (float)W + p.eps);
      ir = 0.5f / sqrtf(s2[1] / (float)W + p.eps);
    }
    const float swt = p.sw ? p.sw[t] : 1.0f;
    float ss = 0.f;
    for (int c = threadIdx.x * V; c < W; c += blockDim.x * V) {
      float v[V];
      if (y2r) {
        float a[V], b[V];
        ldv<T, V>(yr + c, a);
        ldv<T, V>(y2r + c, b);
        if (p.wl) {
          float wa[V], wb[V];
          ldv<float, V>(p.wl + c, wa);
          ldv<float, V>(p.wr + c, wb);
#pragma unroll
          for (int i = 0; i < V; ++i) v[i] = fmaf(a[i] * il, wa[i], b[i] * ir * wb[i]);
        } else {
#pragma unroll
          for (int i = 0; i < V; ++i) v[i] = fmaf(p.cl, a[i], p.cr * b[i]);
        }
      } else if (SLABS) {
        const float* sp = (const float*)p.y + (int64_t)t * W + c;
        if constexpr (V == 4) {
          const f32x4 q = slab_sum<f32x4>(sp, p.slabs, (int64_t)gridDim.x * W);
          v[0] = q[0], v[1] = q[1], v[2] = q[2], v[3] = q[3];
        } else {
          v[0] = slab_sum<float>(sp, p.slabs, (int64_t)gridDim.x * W);
        }
      } else if (yr) {
        ldv<T, V>(yr + c, v);
      } else {
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = 0.f;
        for (int j = 0; j < p.top; ++j) {
          const float wj = p.wts ? p.wts[(int64_t)t * p.top + j] : 1.0f;
          const int pl = p.place[(int64_t)t * p.top + j];
          float e[V];
          if (pl >= 0) ldv<float, V>(p.ey + (int64_t)pl * W + c, e);
          else ldv<T, V>((const T*)p.ident + (int64_t)t * p.ldi + c, e);
#pragma unroll
          for (int i = 0; i < V; ++i) v[i] = fmaf(wj, e[i], v[i]);
        }
        if (sr) {
          float e[V];
          ldv<T, V>(sr + c, e);
#pragma unroll
          for (int i = 0; i < V; ++i) v[i] = fmaf(swt, e[i], v[i]);
        }
      }
      if (rr) {
        float z[V], b[V];
        ldv<T, V>(rr + c, z);
        ldv<float, V>(p.rb + c, b);
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = v[i] / (1.0f + expf(-(z[i] + b[i])));
      }
#pragma unroll
      for (int i = 0; i < V; ++i) {
        buf[c + i] = v[i];
        ss = fmaf(v[i], v[i], ss);
      }
    }
    if (p.groups > 1) {
      part_inv(buf, p);
    } else {
      ss = block_sum(ss, red);
      inv = 1.0f / sqrtf(ss / (float)W + p.eps);
    }
  }
  const float* ar = p.add ? p.add + (int64_t)t * p.lda : nullptr;
  const int part = W / p.groups;
  float ss2 = 0.f;
  for (int c = threadIdx.x * V; c < W; c += blockDim.x * V) {
    float xv[V];
    ldv<float, V>(xr + c, xv);
    if (has_y) {
      float w[V];
      ldv<float, V>(p.wpost + c, w);
#pragma unroll
      for (int i = 0; i < V; ++i) xv[i] = fmaf(buf[c + i] * (p.groups > 1 ? buf[W + (c + i) / part] : inv), w[i], xv[i]);
    }
    if (ar) {
      float a[V];
      ldv<float, V>(ar + c, a);
#pragma unroll
      for (int i = 0; i < V; ++i) xv[i] += a[i];
    }
    if (has_y || ar) stv<float, V>(xr + c, xv);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      buf[c + i] = xv[i];
      ss2 = fmaf(xv[i], xv[i], ss2);
    }
  }
  norm_out<T, V>(buf, ss2, p, t, red);
}

struct SideArgs {
  const int64_t* ids;
  const void* table;  // [vocab, ldt] in the storage type
  int64_t ldt;
  int vocab, col0, d;
  const void* wg;  // [d, W]
  const void* wp;  // [W, d]
  const float* wn;
};

__device__ __forceinline__ float gelu_tanh_f(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// What a row goes through after its closing op, in the same launch (steps of few bf16 rows up to 2048 wide, workgroups of eight waves). A
// decode step is the chain of its launches and of their loads, so a tail's weights are asked for behind the closing op's operands and before
// its first sum.
struct NoTail {
  static constexpr int kind = 0;
};
// the router of the next sublayer's experts, over h as moe_router (moe.hip) has it: the same sums in the same order. Looks of 40 outputs; a second one
// takes longer than a launch of its own, which spreads the outputs over the chip (64 outputs 1.03 - 1.05, 128 1.09 - 1.11 of the time of both),
// so sandwich_add_norm (ops/hip.py) sends no more than 40. (With the loop over looks taken out, 32 outputs over 33 rows took 9.6 us in place of 9.3.)
struct RouteTail {
  static constexpr int kind = 1;
  const bf16_t* wr;  // [E (+ 1), W]
  const float* corr;
  int* idx;
  float* wts;
  int E, top, norm, smax;
  const float* zb;
  float* sg;
};
// the token input (D its numbers, NW at least W / 256), before `add` and the norm. Its weights are asked for under a condition that is the wave's: those
// past a narrow row read again, rows of 256 took 10.4 us for the token input of 64 numbers alone, a kernel of its own before 7.6; now 8.2, and with the
// closing op 0.82 - 0.98 of the two launches at 256 - 2048 (32 numbers 0.82 - 0.87)
template <int D_, int NW_>
struct SideTail : SideArgs {
  static constexpr int kind = 2, D = D_, NW = NW_;
};

// The same for rows of up to 4096 and a norm of one part: a thread keeps NC times four columns of everything in registers, all loads are
// issued before the first sum, and only two sums pass through LDS. The kernel above asks for the stream and the weights behind the
// first sum, a round trip more. us, plain rows / gated / four experts' rows: 33 x 2048 5.0 / 5.3 / 5.5 -> 4.3 / 4.7 / 4.8, 8192 x 2048
// (NT) 48.9 / 58.8 / 88 -> 41.4 / 54.4 / 72.6, 8192 x 1024 24.8 / 28.3 / 37.8 -> 20.6 / 24.5 / 34.1. NT: the stream, y and what is read with it past the caches' replacement.
// With a tail, one launch against two, in a decode step (kernel times, us): the router of 17 outputs over 8 rows of 1024 11.0 -> 7.9, of 32
// over 33 rows of 2048 13.8 -> 11.1, the token input of 32 numbers 17.1 -> 14.7 (each of 33 workgroups draws its 256 KB of weights through one
// CU). A tail's kernel for every form of y at once, its loads behind a branch a column: 8.7, 11.3 and 16.2.
// FORM: what y is, where a launch is a chain that fetches its code as it goes (tails); else found at run time
enum { Y_ANY = -1, Y_NONE, Y_ROWS, Y_SLABS, Y_PAIR, Y_EXPERTS };
template <typename T, int NC, typename TAIL, int FORM, bool NT = false>
__global__ __launch_bounds__(512) void sandwich_rows_kernel(SandwichArgs p, TAIL a) {
  constexpr bool ROUTE = TAIL::kind == 1, SIDE = TAIL::kind == 2;
  static_assert(TAIL::kind == 0 || (NC == 1 && sizeof(T) == 2), "tails: bf16 rows, four columns a thread");
  __shared__ float red[32];
  __shared__ __attribute__((aligned(16))) float row[TAIL::kind == 0 ? 1 : ROUTE ? 1024 + 132 : 2048 + 64];
  const int t = blockIdx.x, W = p.W, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  float* xr = p.x + (int64_t)t * W;
  const int form = FORM != Y_ANY ? FORM : p.y2 ? Y_PAIR : p.slabs ? Y_SLABS : p.y ? Y_ROWS : p.ey ? Y_EXPERTS : Y_NONE;
  const bool has_y = form != Y_NONE;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 x[NC], v[NC], wp[NC], wn[NC], ad[NC];
  int col[NC], at[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    col[i] = 4 * (threadIdx.x + blockDim.x * i);
    at[i] = min(col[i], W - 4);
    x[i] = v[i] = wp[i] = wn[i] = ad[i] = zero;
  }
#define EACH(...)                     \
  _Pragma("unroll") for (int i = 0; i < NC; ++i) \
    if (col[i] < W) {                 \
      __VA_ARGS__;                    \
    }
// loads: threads past the row take its last columns and drop them; as they lie in memory, for a conversion right behind a load waits for it
// before the next one is issued
#define LOAD(...) _Pragma("unroll") for (int i = 0; i < NC; ++i) { __VA_ARGS__; }
  typedef typename std::conditional<sizeof(T) == 2, u16x4, f32x4>::type Raw;
  auto raw = [](const void* q, int64_t o) {
    const Raw* r = reinterpret_cast<const Raw*>((const T*)q + o);
    return NT ? __builtin_nontemporal_load(r) : *r;
  };
  auto wide = [](const float* q) {
    const f32x4* r = reinterpret_cast<const f32x4*>(q);
    return NT ? __builtin_nontemporal_load(r) : *r;
  };
  auto num = [](const Raw& q) {
    if constexpr (sizeof(T) == 2) return f32x4{bf2f(q[0]), bf2f(q[1]), bf2f(q[2]), bf2f(q[3])};
    else return q;
  };
  // ---- a tail's weights
  constexpr int RO = ROUTE ? 5 : 1, RC = ROUTE ? 4 : 1;  // a wave's outputs wv, wv + 8, .. of the first look; pieces of 512 of the width
  u16x8 rw[RO][RC];
  float rcorr[2] = {0.f, 0.f}, rbias[2] = {0.f, 0.f};
  constexpr int SR = [] { if constexpr (SIDE) return TAIL::D / 8; else return 1; }();  // gate rows of a wave
  constexpr int SW = [] { if constexpr (SIDE) return TAIL::NW; else return 1; }();
  u16x4 sgw[SR][SW];
  u16x8 spw[SIDE ? 4 : 1][SR];
  f32x4 swn = zero;
  bf16_t ser = 0;
  int64_t id = 0;
  int eg = 0;
  auto load_route = [&](int e0) {
    if constexpr (ROUTE) {
#pragma unroll
      for (int n = 0; n < RO; ++n)
#pragma unroll
        for (int u = 0; u < RC; ++u)
          rw[n][u] = *reinterpret_cast<const u16x8*>(a.wr + (int64_t)min(e0 + 8 * n, eg - 1) * W + min(lane * 8 + 512 * u, W - 8));
    }
  };
  auto load_proj = [&]() {
    if constexpr (SIDE) {
      if (SW < 8 && __builtin_amdgcn_readfirstlane(wv) * 256 >= W) return;  // (a wave past a narrow row)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < SR; ++j)
          spw[i][j] = *reinterpret_cast<const u16x8*>((const bf16_t*)a.wp + (int64_t)(at[0] + i) * TAIL::D + 8 * j);
    }
  };
  auto load_tail = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ROUTE) {
      load_route(wv);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (a.corr) rcorr[j] = a.corr[min(lane + 64 * j, a.E - 1)];
        if (a.zb) rbias[j] = a.zb[min(lane + 64 * j, a.E - 1)];
      }
    }
    if constexpr (SIDE) {
#pragma unroll
      for (int r = 0; r < SR; ++r)
#pragma unroll
        for (int k = 0; k < SW; ++k)
          if (k * 256 < W) sgw[r][k] = *reinterpret_cast<const u16x4*>((const bf16_t*)a.wg + (int64_t)(wv * SR + r) * W + k * 256 + lane * 4);
      if constexpr (TAIL::D == 32) load_proj();  // (the deeper form's registers hold one of the two at a time)
      swn = ld4(a.wn + at[0]);
      id = id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id);
      ser = ((const bf16_t*)a.table)[id * a.ldt + a.col0 + wv * SR + min(lane, SR - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (ROUTE) eg = a.E + (a.sg ? 1 : 0);
  if constexpr (SIDE) id = a.ids[t];
  LOAD(x[i] = wide(xr + at[i]))
  if (p.wnext) LOAD(wn[i] = ld4(p.wnext + at[i]))
  if (p.add) LOAD(ad[i] = ld4(p.add + (int64_t)t * p.lda + at[i]))
  if (!has_y) load_tail();
  if (has_y) {
    Raw z[NC];
    f32x4 b[NC];
    LOAD(wp[i] = ld4(p.wpost + at[i]))
    if (p.r) LOAD(z[i] = raw(p.r, (int64_t)t * p.ldr + at[i]); b[i] = ld4(p.rb + at[i]))
    if (form == Y_PAIR) {
      Raw q1[NC], q2[NC];
      f32x4 y2[NC], wa[NC], wb[NC];
      LOAD(q1[i] = raw(p.y, (int64_t)t * p.ldy + at[i]); q2[i] = raw(p.y2, (int64_t)t * p.ldy2 + at[i]))
      if (p.wl) LOAD(wa[i] = ld4(p.wl + at[i]); wb[i] = ld4(p.wr + at[i]))
      load_tail();
      LOAD(v[i] = num(q1[i]); y2[i] = num(q2[i]))
      if (p.wl) {  // two mixers: the root mean square of each row first
        float sl = 0.f, sr = 0.f;
        EACH(for (int e = 0; e < 4; ++e) sl = fmaf(v[i][e], v[i][e], sl), sr = fmaf(y2[i][e], y2[i][e], sr))
        const f32x2 s2 = block_sum2(sl, sr, red);
        const float il = 0.5f / sqrtf(s2[0] / (float)W + p.eps), ir = 0.5f / sqrtf(s2[1] / (float)W + p.eps);
        EACH(for (int e = 0; e < 4; ++e) v[i][e] = fmaf(v[i][e] * il, wa[i][e], y2[i][e] * ir * wb[i][e]))
      } else {
        EACH(for (int e = 0; e < 4; ++e) v[i][e] = fmaf(p.cl, v[i][e], p.cr * y2[i][e]))
      }
    } else if (form == Y_SLABS) {
      f32x4 q[8][NC];
      const int64_t ls = (int64_t)gridDim.x * W;
      const float* sp = (const float*)p.y + (int64_t)t * W;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        LOAD(q[j][i] = ld4(sp + min(j, p.slabs - 1) * ls + at[i]))
      load_tail();
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < p.slabs) LOAD(v[i] += q[j][i])
      for (int j = 8; j < p.slabs; ++j) LOAD(v[i] += ld4(sp + j * ls + at[i]))
    } else if (form == Y_ROWS) {
      Raw q[NC];
      LOAD(q[i] = raw(p.y, (int64_t)t * p.ldy + at[i]))
      load_tail();
      LOAD(v[i] = num(q[i]))
    } else {
      Raw sh[NC];
      if (p.shared_) LOAD(sh[i] = raw(p.shared_, (int64_t)t * p.lds_ + at[i]))
      for (int j0 = 0; j0 < p.top; j0 += 4) {  // four pairs in flight
        f32x4 e[4][NC];
        float wj[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int jj = min(j0 + j, p.top - 1);
          const float* er = p.ey + (int64_t)p.place[(int64_t)t * p.top + jj] * W;
          wj[j] = p.wts ? p.wts[(int64_t)t * p.top + jj] : 1.0f;
          LOAD(e[j][i] = wide(er + at[i]))
        }
        if (j0 == 0) load_tail();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j0 + j >= p.top) continue;
          LOAD(for (int k = 0; k < 4; ++k) v[i][k] = fmaf(wj[j], e[j][i][k], v[i][k]))
        }
      }
      const float swt = p.sw ? p.sw[t] : 1.0f;
      if (p.shared_) LOAD(const f32x4 q = num(sh[i]); for (int e = 0; e < 4; ++e) v[i][e] = fmaf(swt, q[e], v[i][e]))
    }
    if (p.r) LOAD(const f32x4 q = num(z[i]); for (int e = 0; e < 4; ++e) v[i][e] = v[i][e] / (1.0f + expf(-(q[e] + b[i][e]))))
    float ss = 0.f;
    EACH(for (int e = 0; e < 4; ++e) ss = fmaf(v[i][e], v[i][e], ss))
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)W + p.eps);
    EACH(for (int e = 0; e < 4; ++e) x[i][e] = fmaf(v[i][e] * inv, wp[i][e], x[i][e]))
  }
  if constexpr (SIDE) {
    constexpr int D = TAIL::D;
    float* gs = row + 2048;
    EACH(*reinterpret_cast<f32x4*>(row + col[i]) = x[i])
    __syncthreads();
    float acc[SR];
#pragma unroll
    for (int r = 0; r < SR; ++r) acc[r] = 0.f;
#pragma unroll
    for (int k = 0; k < SW; ++k)
      if (k * 256 < W) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(row + k * 256 + lane * 4);
#pragma unroll
        for (int r = 0; r < SR; ++r)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[r] = fmaf(bf2f(sgw[r][k][i]), xv[i], acc[r]);
      }
    if constexpr (D != 32) load_proj();
#pragma unroll
    for (int r = 0; r < SR; ++r) {
      acc[r] = warp_sum(acc[r]);
      if (lane == r) gs[wv * SR + r] = gelu_tanh_f(acc[r]) * bf2f(ser);
    }
    __syncthreads();
    f32x4 y = zero;
    if (col[0] < W) {
#pragma unroll
      for (int j = 0; j < SR; ++j) {
        const f32x4 g0 = *reinterpret_cast<const f32x4*>(gs + 8 * j), g1 = *reinterpret_cast<const f32x4*>(gs + 8 * j + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y[i] = fmaf(bf2f(spw[i][j][e]), g0[e], y[i]);
            y[i] = fmaf(bf2f(spw[i][j][4 + e]), g1[e], y[i]);
          }
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(y[i], y[i], ss);
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)W + p.eps);
    EACH(for (int e = 0; e < 4; ++e) x[i][e] = fmaf(y[e] * inv, swn[e], x[i][e]))
  }
  if (p.add) EACH(for (int e = 0; e < 4; ++e) x[i][e] += ad[i][e])
  if (has_y || p.add || SIDE) EACH(if constexpr (NT) __builtin_nontemporal_store(x[i], reinterpret_cast<f32x4*>(xr + col[i])); else st4(xr + col[i], x[i]))
  if (!p.wnext) return;
  float ss = 0.f;
  EACH(for (int e = 0; e < 4; ++e) ss = fmaf(x[i][e], x[i][e], ss))
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)W + p.eps);
  EACH(f32x4 o; for (int e = 0; e < 4; ++e) o[e] = x[i][e] * inv * wn[i][e]; st4((T*)p.h + (int64_t)t * p.ldh + col[i], o);
       if constexpr (ROUTE) st4((bf16_t*)row + col[i], o))
#undef EACH
#undef LOAD
  if constexpr (ROUTE) {
    float* sc = row + 1024;
    __syncthreads();
    u16x8 hv[RC];
#pragma unroll
    for (int u = 0; u < RC; ++u) hv[u] = *reinterpret_cast<const u16x8*>((const bf16_t*)row + min(lane * 8 + 512 * u, W - 8));
    for (int e0 = wv; e0 < eg; e0 += 8 * RO) {
      if (e0 != wv) load_route(e0);
#pragma unroll
      for (int n = 0; n < RO; ++n) {
        const int e = e0 + 8 * n;
        if (e >= eg) break;
        float z = 0.f;
#pragma unroll
        for (int u = 0; u < RC; ++u) {
          if (lane * 8 + 512 * u >= W) break;
#pragma unroll
          for (int i = 0; i < 8; ++i) z = fmaf(bf2f(hv[u][i]), bf2f(rw[n][u][i]), z);
        }
        z = warp_sum(z);
        if (lane != 0) continue;
        if (e == a.E) a.sg[t] = 1.f / (1.f + expf(-z));
        else sc[e] = z;
      }
    }
    __syncthreads();
    if (wv) return;
    float z[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) z[j] = lane + 64 * j < a.E ? sc[lane + 64 * j] + rbias[j] : -INFINITY;
    __builtin_amdgcn_wave_barrier();
    route_ranked(z, sc, rcorr, a.idx + (int64_t)t * a.top, a.wts + (int64_t)t * a.top, a.E, a.top, a.norm, a.smax);
  }
}

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

struct SandwichTail {
  int kind;  // 0: none, 1: route, 2: side
  RouteTail route;
  SideArgs side;
};

template <typename TAIL>
static void launch_tail(const SandwichArgs& p, const TAIL& a, int T_, hipStream_t st) {
  if (p.y2) sandwich_rows_kernel<bf16_t, 1, TAIL, Y_PAIR><<<T_, 512, 0, st>>>(p, a);
  else if (p.slabs) sandwich_rows_kernel<bf16_t, 1, TAIL, Y_SLABS><<<T_, 512, 0, st>>>(p, a);
  else if (p.y) sandwich_rows_kernel<bf16_t, 1, TAIL, Y_ROWS><<<T_, 512, 0, st>>>(p, a);
  else if (p.ey) sandwich_rows_kernel<bf16_t, 1, TAIL, Y_EXPERTS><<<T_, 512, 0, st>>>(p, a);
  else sandwich_rows_kernel<bf16_t, 1, TAIL, Y_NONE><<<T_, 512, 0, st>>>(p, a);
}

// rows a token input can follow in the closing op's launch
static bool side_tail_ok(const SideArgs& s, int W) {
  return (s.d == 32 || s.d == 64) && W % 256 == 0 && W <= 2048 && al16(s.wp) && al16(s.wn) && ((uintptr_t)s.wg & 7) == 0;
}
static void launch_side_tail(const SandwichArgs& p, const SideArgs& s, int T_, hipStream_t st) {
  if (!side_tail_ok(s, p.W)) throw std::runtime_error("sandwich_add_norm: token input of 32 or 64 numbers over aligned rows of whole 256s");
#define LAUNCH_ROW(D_, NW_) launch_tail(p, SideTail<D_, NW_>{s}, T_, st)
  if (s.d == 32 && p.W <= 1024) LAUNCH_ROW(32, 4);
  else if (s.d == 32) LAUNCH_ROW(32, 8);
  else if (p.W <= 1024) LAUNCH_ROW(64, 4);
  else LAUNCH_ROW(64, 8);
#undef LAUNCH_ROW
}

static void launch_sandwich_add_norm(void* x, const void* y, int64_t ldy, const void* ey, const void* place, const void* wts,
                              int top, const void* shared_, int64_t lds_, const void* r, int64_t ldr, const void* rb,
                              const void* wpost, const void* add, const void* wnext, void* h, int64_t ldh, float eps,
                              int groups, const void* ident, int64_t ldi, const void* y2, int64_t ldy2, const void* wl,
                              const void* wr, float cl, float cr, int64_t lda, const void* sw, int slabs, int T_, int W, int dt,
                              const SandwichTail& tail, hipStream_t st) {
  if (T_ == 0) return;
  if (groups < 1 || W % groups) throw std::runtime_error("sandwich_add_norm: the norm's parts must divide the row");
  if (((size_t)W + groups) * 4 > 64 * 1024) throw std::runtime_error("sandwich_add_norm: rows wider than 16384");
  SandwichArgs p{(float*)x, y, ldy, (const float*)ey, (const int*)place, (const float*)wts, top, shared_, lds_, r, ldr,
                 (const float*)rb, (const float*)wpost, (const float*)add, (const float*)wnext, h, ldh, eps, W, groups, ident, ldi, y2, ldy2,
                 (const float*)wl, (const float*)wr, cl, cr, lda, (const float*)sw, slabs};
  const int es = dt == 0 ? 2 : 4;
  const auto alv = [&](const void* q, int64_t ld) { return !q || (((uintptr_t)q % (4 * es)) == 0 && ld % 4 == 0); };
  const bool vec = W % 4 == 0 && (!slabs || al16(y)) && al16(x) && al16(ey) && al16(rb) && al16(wpost) && al16(add) && al16(wnext) &&
                   alv(y, ldy) && alv(shared_, lds_) && alv(r, ldr) && alv(h, ldh) && alv(ident, ldi) && alv(y2, ldy2) &&
                   al16(wl) && al16(wr);
  const size_t lds = ((size_t)W + (groups > 1 ? groups : 0)) * 4;
  const int th = T_ <= 512 && W > 1024 ? 512 : 256;  // few rows: more waves to a row
  // (identity experts and norms in parts keep the general kernel, and so do rows wider than 1280 without y, 2048 x 8192 24.3 and 25.8, from
  // 1025 to 2048 of them with it, 1500 x 2048 13.6 and 14.7, and many wider than 2048, 8192 x 4096 83.7 and 89.1 us. 4096 x 2048 plain 21.8 ->
  // 20.1, gated 30.9 -> 27.4, 8192 rows 48.9 -> 44.3 and 58.8 -> 59.6, past the caches 41.4 and 54.4)
  const bool rows = vec && groups == 1 && !ident && (W <= 1280 || (W <= 2048 && (T_ <= 1024 || ((y || ey) && T_ > 2048))) || (W <= 4096 && T_ <= 512));
  // a stream that the caches do not keep until the next closing op passes their replacement by, with what is read beside it: also four experts'
  // rows, 8192 x 2048, 88 -> 72.6; but 8192 x 1024, 34 MB, 20.1 -> 22.7. With the two products of a feed-forward behind it, rows of 1024 - 2048:
  // streams of 48 - 200 MB 0.965 - 1.007 of the time, experts' 0.91 - 0.975, of 24 - 42 MB to 1.016
  const bool past = (y || ey) && (int64_t)T_ * W * 4 >= (48 << 20);
  if (slabs < 0 || (slabs && (!y || y2))) throw std::runtime_error("sandwich_add_norm: slabs of one product only");
  if (tail.kind) {
    if (!vec || groups != 1 || ident || dt != 0 || W > 2048) throw std::runtime_error("sandwich_add_norm: a tail needs whole bf16 rows of up to 2048 at aligned places");
    if (tail.kind == 1) {
      const RouteTail& r_ = tail.route;
      if (!wnext || W % 8 || !al16(r_.wr) || r_.E < 1 || r_.E > 128 || r_.top < 1 || r_.top > r_.E)
        throw std::runtime_error("sandwich_add_norm: router of 1 - 128 outputs over aligned rows");
      launch_tail(p, r_, T_, st);
    } else {
      launch_side_tail(p, tail.side, T_, st);
    }
    HIP_CHECK_LAUNCH();
    return;
  }
  // whole waves, no more than the row has columns for (256 and 512 threads: 1600 rows and more of 256 1.44, of 1280 1.11 times as long), but for
  // 448, which spread unevenly over the SIMDs (1792 wide: 1.07)
  const int rth = W <= 1536 ? (W / 4 + 63) / 64 * 64 : 512;
  DISPATCH_T(dt, T, {
    if (rows && W <= 2048 && past) sandwich_rows_kernel<T, 1, NoTail, Y_ANY, true><<<T_, rth, 0, st>>>(p, NoTail{});
    else if (rows && W <= 2048) sandwich_rows_kernel<T, 1, NoTail, Y_ANY><<<T_, rth, 0, st>>>(p, NoTail{});
    else if (rows) sandwich_rows_kernel<T, 2, NoTail, Y_ANY><<<T_, 512, 0, st>>>(p, NoTail{});
    else if (slabs && vec) sandwich_add_norm_kernel<T, 4, true><<<T_, th, lds, st>>>(p);
    else if (slabs) sandwich_add_norm_kernel<T, 1, true><<<T_, th, lds, st>>>(p);
    else if (vec) sandwich_add_norm_kernel<T, 4><<<T_, th, lds, st>>>(p);
    else sandwich_add_norm_kernel<T, 1><<<T_, th, lds, st>>>(p);
  });
  HIP_CHECK_LAUNCH();
}

// buf: [W] the x row, then [W] the projected row, then [d] the gated numbers
template <typename T, int V>
__global__ __launch_bounds__(512) void token_side_add_kernel(SandwichArgs p, SideArgs s) {
  extern __shared__ __attribute__((aligned(16))) float buf[];
  __shared__ float red[16];
  const int t = blockIdx.x, W = p.W, d = s.d;
  float* xs = buf;
  float* ys = buf + W;
  float* gs = ys + W;
  float* xr = p.x + (int64_t)t * W;
  for (int c = threadIdx.x * V; c < W; c += blockDim.x * V) {
    float v[V];
    ldv<float, V>(xr + c, v);
#pragma unroll
    for (int i = 0; i < V; ++i) xs[c + i] = v[i];
  }
  __syncthreads();
  int64_t id = s.ids[t];
  id = id < 0 ? 0 : (id >= s.vocab ? s.vocab - 1 : id);
  const T* er = (const T*)s.table + id * s.ldt + s.col0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int j = wv; j < d; j += nw) {  // a wave per gate row, lanes over the width
    const T* wr = (const T*)s.wg + (int64_t)j * W;
    float a = 0.f;
    for (int c = lane * V; c < W; c += 64 * V) {
      float w[V];
      ldv<T, V>(wr + c, w);
#pragma unroll
      for (int i = 0; i < V; ++i) a = fmaf(w[i], xs[c + i], a);
    }
    a = warp_sum(a);
    if (lane == 0) gs[j] = gelu_tanh_f(a) * El<T>::ld(er + j);
  }
  __syncthreads();
  float ss = 0.f;
  const bool rows16 = sizeof(T) == 2 && d % 8 == 0 && ((uintptr_t)s.wp & 15) == 0;  // 16-byte reads of a bf16 row
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const T* wr = (const T*)s.wp + (int64_t)c * d;
    float a = 0.f, a2 = 0.f;
    if (rows16) {
      for (int j = 0; j < d; j += 8) {
        const u16x8 w8 = *reinterpret_cast<const u16x8*>(wr + j);
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          a = fmaf(bf2f(w8[i]), gs[j + i], a);
          a2 = fmaf(bf2f(w8[i + 1]), gs[j + i + 1], a2);
        }
      }
      a += a2;
    } else {
      for (int j = 0; j < d; ++j) a = fmaf(El<T>::ld(wr + j), gs[j], a);
    }
    ys[c] = a;
    ss = fmaf(a, a, ss);
  }
  ss = block_sum(ss, red);  // (its barriers also make ys visible)
  const float inv = 1.0f / sqrtf(ss / (float)W + p.eps);
  const float* ar = p.add ? p.add + (int64_t)t * W : nullptr;
  float ss2 = 0.f;
  for (int c = threadIdx.x * V; c < W; c += blockDim.x * V) {
    float xv[V], w[V];
    ldv<float, V>(s.wn + c, w);
#pragma unroll
    for (int i = 0; i < V; ++i) xv[i] = fmaf(ys[c + i] * inv, w[i], xs[c + i]);
    if (ar) {
      float a[V];
      ldv<float, V>(ar + c, a);
#pragma unroll
      for (int i = 0; i < V; ++i) xv[i] += a[i];
    }
    stv<float, V>(xr + c, xv);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      xs[c + i] = xv[i];
      ss2 = fmaf(xv[i], xv[i], ss2);
    }
  }
  norm_out<T, V>(xs, ss2, p, t, red);
}

// The token input for bf16 weights, 16 rows per workgroup on the matrix cores (the kernel above reads both small matrices from L2
// for every row: 2 GB per prompt step
// of 8192 rows at width 2048, 189 us; 52 us here, of which 27 are the bytes of x and h: a workgroup is a chain of two products and
// two norms of 25 us, so below 1024 rows, where the chip is not filled twice, the kernels above are the faster ones). Wave w takes an eighth of the width. First product:
// the fp32 rows enter as three bf16 numbers that add up to them exactly, the weights are exact, the waves' sums meet in LDS.
// Second: the weights' rows are the first operand, so that a lane holds four neighbouring columns of one row - 16-byte accesses
// of x, 8-byte ones of h - and the projected row, then the new x, stay in registers between the norms.
// DT: 16-number blocks of d; NT: 16-column blocks per wave, at least W / 128. FILL: as many, and then without a question for each block (8192 rows of
// 2048 53.0 -> 52.3 us, 2777 28.1 -> 27.3, 8192 of 4096 with 64 numbers 182 -> 163).
template <int DT, int NT, bool FILL>
__global__ __launch_bounds__(512, NT <= 16 ? 4 : 2) void token_side_rows_kernel(SandwichArgs p, SideArgs s, int T_) {
  constexpr int D = 16 * DT, LDG = D + 4;
  __shared__ __attribute__((aligned(16))) float part[8 * 16 * D];
  __shared__ __attribute__((aligned(16))) float gs[16 * LDG];
  __shared__ float red[2][8 * 16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16, W = FILL ? 128 * NT : p.W, span = W >> 3, c0 = w * span;
  const int t = min(t0 + li, T_ - 1);  // this lane's row, as first operand and in the results
  const bf16_t* wg = (const bf16_t*)s.wg;
  const bf16_t* wp = (const bf16_t*)s.wp;
  float* xr = p.x + (int64_t)t * W;
  auto split = [](const float* v, s16x8& h, s16x8& m, s16x8& l) {
#pragma unroll
    for (int i = 0; i < 8; ++i) split3(v[i], i, h, m, l);
  };
  f32x4 acc[DT];
#pragma unroll
  for (int k = 0; k < DT; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = c0 + 8 * g; k < c0 + span; k += 32) {
    float v[8];
    ldv<float, 4>(xr + k, v);
    ldv<float, 4>(xr + k + 4, v + 4);
    s16x8 b[DT], h, m, l;
#pragma unroll
    for (int j = 0; j < DT; ++j) b[j] = *reinterpret_cast<const s16x8*>(wg + (int64_t)(16 * j + li) * W + k);
    split(v, h, m, l);
#pragma unroll
    for (int j = 0; j < DT; ++j) {
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, b[j], acc[j], 0, 0, 0);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(m, b[j], acc[j], 0, 0, 0);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, b[j], acc[j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < DT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) part[(w * 16 + 4 * g + i) * D + 16 * j + li] = acc[j][i];
  __syncthreads();
  for (int e = tid; e < 16 * D; e += 512) {
    const int r = e / D, j = e - r * D;
    float a = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) a += part[(k * 16 + r) * D + j];
    int64_t id = s.ids[min(t0 + r, T_ - 1)];
    id = id < 0 ? 0 : (id >= s.vocab ? s.vocab - 1 : id);
    gs[r * LDG + j] = gelu_tanh_f(a) * bf2f(((const bf16_t*)s.table)[id * s.ldt + s.col0 + j]);
  }
  __syncthreads();
  f32x4 y[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) y[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < DT / 2; ++k) {
    float v[8];
    s16x8 h, m, l;
    ldv<float, 4>(&gs[li * LDG + 32 * k + 8 * g], v);
    ldv<float, 4>(&gs[li * LDG + 32 * k + 8 * g + 4], v + 4);
    split(v, h, m, l);
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      // (blocks past the wave's columns take its last one again; their sums are dropped below)
      const s16x8 a = *reinterpret_cast<const s16x8*>(wp + (int64_t)(c0 + min(16 * ct, span - 16) + li) * D + 32 * k + 8 * g);
      y[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, l, y[ct], 0, 0, 0);
      y[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, m, y[ct], 0, 0, 0);
      y[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, h, y[ct], 0, 0, 0);
    }
  }
  auto row_inv = [&](float ss, float* r8) {  // 1 / root mean square of the lane's row
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (g == 0) r8[w * 16 + li] = ss;
    __syncthreads();
    float a = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) a += r8[k * 16 + li];
    return 1.0f / sqrtf(a / (float)W + p.eps);
  };
  float ss = 0.f;
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    if (16 * ct >= span) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(y[ct][i], y[ct][i], ss);
  }
  const float inv = row_inv(ss, red[0]);
  const bool in = t0 + li < T_;
  const float* ar = p.add ? p.add + (int64_t)t * W : nullptr;
  ss = 0.f;
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    if (16 * ct >= span) continue;
    const int c = c0 + 16 * ct + 4 * g;
    float xv[4], wn[4];
    ldv<float, 4>(xr + c, xv);
    ldv<float, 4>(s.wn + c, wn);
#pragma unroll
    for (int i = 0; i < 4; ++i) xv[i] = fmaf(y[ct][i] * inv, wn[i], xv[i]);
    if (ar) {
      float a[4];
      ldv<float, 4>(ar + c, a);
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[i] += a[i];
    }
    if (in) stv<float, 4>(xr + c, xv);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[ct][i] = xv[i];
      ss = fmaf(xv[i], xv[i], ss);
    }
  }
  if (!p.wnext) return;
  const float inv2 = row_inv(ss, red[1]);
  bf16_t* hr = (bf16_t*)p.h + (int64_t)t * p.ldh;
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    if (16 * ct >= span) continue;
    const int c = c0 + 16 * ct + 4 * g;
    float wn[4], o[4];
    ldv<float, 4>(p.wnext + c, wn);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = y[ct][i] * inv2 * wn[i];
    if (in) stv<bf16_t, 4>(hr + c, o);
  }
}

void launch_token_side_add(void* x, const void* ids, const void* table, int64_t ldt, int vocab, int col0, int d,
                           const void* wg, const void* wp, const void* wn, const void* add, const void* wnext, void* h,
                           int64_t ldh, float eps, int T_, int W, int dt, hipStream_t st) {
  if (T_ == 0) return;
  const size_t lds = ((size_t)2 * W + d) * 4;
  if (lds > 64 * 1024) throw std::runtime_error("token_side_add: rows too wide");
  SandwichArgs p{};
  p.x = (float*)x; p.add = (const float*)add; p.wnext = (const float*)wnext; p.h = h; p.ldh = ldh; p.eps = eps; p.W = W; p.groups = 1;
  SideArgs s{(const int64_t*)ids, table, ldt, vocab, col0, d, wg, wp, (const float*)wn};
  const int es = dt == 0 ? 2 : 4;
  const bool vec = W % 4 == 0 && al16(x) && al16(wn) && al16(add) && al16(wnext) && ((uintptr_t)wg % (4 * es)) == 0 &&
                   (!h || (((uintptr_t)h % (4 * es)) == 0 && ldh % 4 == 0));
  if (dt == 0 && vec && T_ >= 1024 && (d == 32 || d == 64) && W % 256 == 0 && W <= 4096 && al16(wg) && al16(wp)) {
#define LAUNCH_SIDE1(DT_, NT_)                                                                                     \
  do {                                                                                                            \
    if (W == 128 * NT_) token_side_rows_kernel<DT_, NT_, true><<<(T_ + 15) / 16, 512, 0, st>>>(p, s, T_);         \
    else token_side_rows_kernel<DT_, NT_, false><<<(T_ + 15) / 16, 512, 0, st>>>(p, s, T_);                       \
  } while (0)
#define LAUNCH_SIDE(DT_)                     \
  do {                                       \
    if (W <= 1024) LAUNCH_SIDE1(DT_, 8);     \
    else if (W <= 2048) LAUNCH_SIDE1(DT_, 16); \
    else LAUNCH_SIDE1(DT_, 32);              \
  } while (0)
    if (d == 32) LAUNCH_SIDE(2);
    else LAUNCH_SIDE(4);
#undef LAUNCH_SIDE
#undef LAUNCH_SIDE1
    HIP_CHECK_LAUNCH();
    return;
  }
  // (a row per workgroup, everything it needs asked for at the start: 33 rows of 2048 in a decode step 24 -> 15 us. A CU holds one
  // workgroup: up to 256 rows (12.6 us), at 1006 it takes 43 us and the kernel above 26.)
  if (dt == 0 && vec && T_ <= 256 && side_tail_ok(s, W)) {
    p.lda = W;
    launch_side_tail(p, s, T_, st);
    HIP_CHECK_LAUNCH();
    return;
  }
  DISPATCH_T(dt, T, {
    if (vec) token_side_add_kernel<T, 4><<<T_, 512, lds, st>>>(p, s);
    else token_side_add_kernel<T, 1><<<T_, 512, lds, st>>>(p, s);
  });
  HIP_CHECK_LAUNCH();
}

void launch_sandwich_tail(void* x, const void* y, int64_t ldy, const void* ey, const void* place, const void* wts, int top,
                          const void* shared_, int64_t lds_, const void* r, int64_t ldr, const void* rb, const void* wpost,
                          const void* add, const void* wnext, void* h, int64_t ldh, float eps, const void* y2, int64_t ldy2,
                          const void* wl, const void* wr, float cl, float cr, int64_t lda, const void* sw, int slabs, int T_, int W,
                          int kind, const void* router, const void* corr, void* idx, void* rwts, int E, int rtop, int norm, int smax,
                          const void* zb, void* sg, const void* ids, const void* table, int64_t ldt, int vocab, int col0, int d,
                          const void* wg, const void* wp, const void* wn, hipStream_t st) {
  SandwichTail t{kind};
  if (kind == 1) {
    t.route.wr = (const bf16_t*)router, t.route.corr = (const float*)corr, t.route.idx = (int*)idx, t.route.wts = (float*)rwts;
    t.route.E = E, t.route.top = rtop, t.route.norm = norm, t.route.smax = smax;
    t.route.zb = (const float*)zb, t.route.sg = (float*)sg;
  } else if (kind == 2) {
    t.side = SideArgs{(const int64_t*)ids, table, ldt, vocab, col0, d, wg, wp, (const float*)wn};
  } else {
    throw std::runtime_error("sandwich_tail: kind");
  }
  launch_sandwich_add_norm(x, y, ldy, ey, place, wts, top, shared_, lds_, r, ldr, rb, wpost, add, wnext, h, ldh, eps, 1, nullptr, 0, y2,
                           ldy2, wl, wr, cl, cr, lda, sw, slabs, T_, W, 0, t, st);
}

void launch_sandwich_add_norm(void* x, const void* y, int64_t ldy, const void* ey, const void* place, const void* wts,
                              int top, const void* shared_, int64_t lds_, const void* r, int64_t ldr, const void* rb,
                              const void* wpost, const void* add, const void* wnext, void* h, int64_t ldh, float eps,
                              int groups, const void* ident, int64_t ldi, const void* y2, int64_t ldy2, const void* wl,
                              const void* wr, float cl, float cr, int64_t lda, const void* sw, int slabs, int T_, int W, int dt,
                              hipStream_t st) {
  launch_sandwich_add_norm(x, y, ldy, ey, place, wts, top, shared_, lds_, r, ldr, rb, wpost, add, wnext, h, ldh, eps, groups, ident, ldi,
                           y2, ldy2, wl, wr, cl, cr, lda, sw, slabs, T_, W, dt, SandwichTail{}, st);
}
