// Grouped expert products of a few rows per expert (decode steps; bf16).
//
// Bound by the experts' weights, each read once: a step of 33 tokens over 32 experts of 2048 x 768 reads 300 MB. A workgroup takes two
// groups of 16 weight rows - 16 gate and their 16 up rows, or 32 rows of one matrix - against a tile's rows; its four waves
// split K and meet in LDS, and a wave asks for four steps of 64 at once (24 KB in flight a wave) straight into the matrix
// instructions' operands: no staging, no barrier before the end. The 64-row tiles that larger steps
// take keep one step of 64 in flight and four waves behind barriers.
// All products of a layer, weights from memory, against those (us): 32 experts of 2048 x 768, 4 rows each, 81 -> 75; 16 of 1024 x 512
// 37 -> 25; 8 of 4096 x 2048 120 -> 86, one row each 110 -> 63. A tile more for an expert reads its weights again.
// Whole lines past the caches' replacement (md_products64) against half lines of 16 rows: 217 MB of gate and up rows (33 tokens, 32 experts and a
// shared one) 53 -> 40 us, 5.4 TB/s, 105 MB of down rows 31.5 -> 25.8; reads alone, 210 MB, 36.9 and 32.5 us, half lines past the caches 38.3.
//
// Who chose whom: up to MD_PAIRS (token, expert) pairs a workgroup finds its expert's pairs itself, with one look at all choices, and the
// rows of the results are the pairs' own numbers: no grouping launch before the products. With fewer pairs than experts there is a workgroup row a
// pair, and an expert's first pair has it: with one an expert, most of which found nobody, 60 experts of 192 x 832 took 20.9 us for 8
// pairs, 14.7 with a grouping launch, and 384 of 2368 x 320 took 73 for 4, 33 with it. Beyond that, or where the workgroups that find nothing cost more than the launch, it reads moe.hip's tile list, 16 rows a tile. The shared expert's products, and
// columns of further weights behind its gate and up rows, ride along as workgroups of their own, 32 rows each.
// A layer's experts in a decode step, grouping and the shared expert's launches beside them before: 33 rows, 32 experts of 2048 x 768 and a
// shared one of 1024 with 2048 further columns, 14 us less; 8 rows, 16 experts of 1024 x 512 and a shared one of 512, 11 us less.
#include <cmath>

#include "anytype.h"
#include "gemm_quad.h"

enum { MD_GLU = 0, MD_GELU = 1, MD_DOWN = 2 };
#define MD_PAIRS 1024  // a look of four numbers a thread
#define MD_ROWS 32     // rows of a tile found that way

struct MoeDecArgs {
  const bf16_t* X;
  int64_t ldx;
  const bf16_t* W;   // gate (MD_GLU), up (MD_GELU) or down
  const bf16_t* W2;  // MD_GLU: up; null: gate and up rows of W in alternating groups of 16
  void* C;           // [pairs, N]: bf16, MD_DOWN fp32
  int N, K;
  const int* meta;   // LIST: the tile list and the pair of every row
  const int* order;
  const float* pw;   // weights on the inputs, or null
  int E, maxt, top, silu;
  float limit, alpha;
  // not LIST
  const int* idx;  // [P] the pairs' experts
  int* place;      // (MD_DOWN: null) [P] row of a pair's result: the pair, or -1 for an expert that is none
  int P, xt;       // pairs; workgroups for experts of more than MD_ROWS pairs
  int T;           // the shared expert's rows (0: none)
  const bf16_t* sX;  // MD_DOWN: its activations
  const bf16_t* sW;  // gate rows, then up rows (or alternating groups of 16), then sE further rows; MD_DOWN: [N, sK]
  bf16_t* sC;        // MD_GLU: activations [T, sN]; MD_DOWN: [T, N]
  bf16_t* sD;        // the further rows' results
  int64_t sldd;
  int sN, sK, sE, sinter;
  float slimit;
};

// G groups of 16 rows against the two groups of weight rows, steps [s, s1) of 64: a load takes whole lines, 128 bytes of eight rows (lane l: piece
// l / 8 of row l % 8), past the caches' replacement - every weight is read once. The matrix instructions want 16 rows side by side: of two
// such loads, lanes 0 - 7 and 8 - 15 of every 16 change places, and lane (li, g) holds pieces 2 g and 2 g + 1 of row li. wa: this lane's place
// in rows 0 - 7 and in rows 8 - 15
template <int G, int U>
__device__ __forceinline__ void md_products64(const bf16_t* const (&wa)[2], const bf16_t* const (&wb)[2], const bf16_t* const (&x)[G], int s,
                                              int s1, f32x4 (&aa)[G], f32x4 (&ab)[G]) {
#pragma unroll
  for (int q = 0; q < G; ++q) aa[q] = ab[q] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto turn = [](const s16x8& lo, const s16x8& hi, s16x8& even, s16x8& odd) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4 l = __builtin_bit_cast(i32x4, lo), h = __builtin_bit_cast(i32x4, hi);
    i32x4 e, o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      e[i] = __builtin_amdgcn_update_dpp(l[i], h[i], 0x128, 0xf, 0xc, false);  // (the row of 16 turned by 8, into its lanes 8 - 15)
      o[i] = __builtin_amdgcn_update_dpp(h[i], l[i], 0x128, 0xf, 0x3, false);
    }
    even = __builtin_bit_cast(s16x8, e), odd = __builtin_bit_cast(s16x8, o);
  };
  for (; s < s1; s += U) {
    s16x8 fx[G][U][2], fa[U][2], fb[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + u, s1 - 1) * 64;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[u][i] = __builtin_nontemporal_load(reinterpret_cast<const s16x8*>(wa[i] + k));
        fb[u][i] = __builtin_nontemporal_load(reinterpret_cast<const s16x8*>(wb[i] + k));
#pragma unroll
        for (int q = 0; q < G; ++q) fx[q][u][i] = *reinterpret_cast<const s16x8*>(x[q] + k + 8 * i);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s1) {
        s16x8 a0, a1, b0, b1;
        turn(fa[u][0], fa[u][1], a0, a1);
        turn(fb[u][0], fb[u][1], b0, b1);
#pragma unroll
        for (int q = 0; q < G; ++q) {
          aa[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, fx[q][u][0], aa[q], 0, 0, 0);
          ab[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, fx[q][u][0], ab[q], 0, 0, 0);
          aa[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, fx[q][u][1], aa[q], 0, 0, 0);
          ab[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, fx[q][u][1], ab[q], 0, 0, 0);
        }
      }
  }
}

// The same in steps of 32, straight in the operands' places (K no multiple of 64)
template <int G, int U>
__device__ __forceinline__ void md_products(const bf16_t* wa, const bf16_t* wb, const bf16_t* const (&x)[G], int s, int s1, f32x4 (&aa)[G],
                                            f32x4 (&ab)[G]) {
#pragma unroll
  for (int q = 0; q < G; ++q) aa[q] = ab[q] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (; s < s1; s += U) {
    s16x8 fx[G][U], fa[U], fb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + u, s1 - 1) * 32;
      fa[u] = *reinterpret_cast<const s16x8*>(wa + k);
      fb[u] = *reinterpret_cast<const s16x8*>(wb + k);
#pragma unroll
      for (int q = 0; q < G; ++q) fx[q][u] = *reinterpret_cast<const s16x8*>(x[q] + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s1) {
#pragma unroll
        for (int q = 0; q < G; ++q) {
          aa[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[u], fx[q][u], aa[q], 0, 0, 0);
          ab[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[u], fx[q][u], ab[q], 0, 0, 0);
        }
      }
  }
}

// The expert that the workgroup `j` of those for tiles past an expert's first takes, and which of its tiles: {expert, tile}, or {-1, 0}
__device__ __forceinline__ int2 md_extra(const MoeDecArgs& p, int j, int* cnt) {
  __shared__ int2 found;
  for (int e = threadIdx.x; e < p.E; e += 256) cnt[e] = 0;
  if (threadIdx.x == 0) found = int2{-1, 0};
  __syncthreads();
  for (int q = threadIdx.x; q < p.P; q += 256) {
    const int e = p.idx[q];
    if ((unsigned)e < (unsigned)p.E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    int before = 0;
    for (int e0 = 0; e0 < p.E; e0 += 64) {
      const int e = e0 + threadIdx.x, c = e < p.E ? max(0, (cnt[e] - 1) / MD_ROWS) : 0;
      int sum = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(sum, d, 64);
        sum += (int)threadIdx.x >= d ? o : 0;
      }
      const int at = j - (before + sum - c);
      if (at >= 0 && at < c) found = int2{e, at + 1};
      before += __shfl(sum, 63, 64);
    }
  }
  __syncthreads();
  return found;
}

// WHO: a tile's rows from moe.hip's tile list, or found here, a workgroup row an expert or (fewer of them) a pair
enum { WHO_LIST, WHO_EXPERT, WHO_PAIR };
template <int MODE, int WHO, bool LINES>
__global__ __launch_bounds__(256, 4) void moe_dec_kernel(MoeDecArgs p) {
  constexpr bool LIST = WHO == WHO_LIST;
  constexpr int BN = MODE == MD_GLU ? 16 : 32, G = LIST ? 1 : 2;
  __shared__ __attribute__((aligned(16))) float part[4][2][16 * G][20];  // (rows of 20: 16-byte places, spread over the banks)
  __shared__ int list[MD_ROWS], found[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  int K = p.K, N = p.N, rows, row0 = 0, n0;
  bool shared_ = false, plain = MODE != MD_GLU, inter = MODE == MD_GLU && !p.W2;
  int64_t ldx = p.ldx;
  const bf16_t *x, *W = p.W, *W2 = p.W2;
  if constexpr (LIST) {
    if ((int)blockIdx.y >= p.meta[0]) return;
    const int e = p.meta[1 + (p.E + 1) + blockIdx.y];
    row0 = p.meta[1 + (p.E + 1) + p.maxt + blockIdx.y];
    rows = min(16, p.meta[1 + e + 1] - row0);
    n0 = blockIdx.x * BN;
    x = p.X;
    W += (int64_t)e * (MODE == MD_GLU && !W2 ? 2 : 1) * N * K;
    if (W2) W2 += (int64_t)e * N * K;
  } else {
    if (MODE != MD_DOWN && blockIdx.x == 0)
      for (int q = threadIdx.x; q < p.P; q += 256) p.place[q] = (unsigned)p.idx[q] < (unsigned)p.E ? q : -1;
    const int st = (p.T + MD_ROWS - 1) / MD_ROWS, sg = ((MODE == MD_GLU ? p.sN : p.N) + BN - 1) / BN;
    const int sb = st * (sg + (p.sE + 31) / 32);  // workgroups of the shared expert, a column's row tiles side by side
    int b = blockIdx.x;
    if (b < sb) {
      shared_ = true;
      row0 = b % st * MD_ROWS;
      rows = min(MD_ROWS, p.T - row0);
      const int c = b / st;
      x = MODE == MD_DOWN ? p.sX : p.X;
      K = p.sK, W = p.sW, inter = p.sinter;
      if (MODE == MD_DOWN) ldx = p.sK, n0 = c * BN;
      else if (c < sg) N = p.sN, n0 = c * BN, W2 = inter ? nullptr : W + (int64_t)N * K;
      else plain = true, n0 = (c - sg) * 32, N = p.sE, W += (int64_t)2 * p.sN * K;
    } else {
      b -= sb;
      const int ct = (N + BN - 1) / BN;
      int e = b / ct, tile = 0, pair = -1;
      n0 = b % ct * BN;
      const int firsts = WHO == WHO_PAIR ? p.P : p.E;
      if (e >= firsts) {
        const int2 f = md_extra(p, e - firsts, reinterpret_cast<int*>(part));
        if (f.x < 0) return;
        e = f.x, tile = f.y;
      } else if constexpr (WHO == WHO_PAIR) {
        pair = e;
        e = p.idx[pair];
        if ((unsigned)e >= (unsigned)p.E) return;
      }
      // the expert's pairs, by number: each wave counts those of its 64 numbers
      int v[MD_PAIRS / 256];
      unsigned long long m[MD_PAIRS / 256];
#pragma unroll
      for (int u = 0; u < MD_PAIRS / 256; ++u) v[u] = (int)threadIdx.x + 256 * u < p.P ? p.idx[threadIdx.x + 256 * u] : -1;
#pragma unroll
      for (int u = 0; u < MD_PAIRS / 256; ++u) {
        m[u] = __ballot(v[u] == e);
        if (lane == 0) found[4 * u + w] = __popcll(m[u]);
      }
      __syncthreads();
      int total = 0, before[MD_PAIRS / 256];
#pragma unroll
      for (int i = 0; i < MD_PAIRS / 64; ++i) {
        if ((i & 3) == w) before[i >> 2] = total;
        total += found[i];
      }
      rows = min(MD_ROWS, total - MD_ROWS * tile);
      if (rows <= 0) return;
#pragma unroll
      for (int u = 0; u < MD_PAIRS / 256; ++u) {
        const int r = before[u] + __popcll(m[u] & ((1ull << lane) - 1)) - MD_ROWS * tile;
        if (v[u] == e && r >= 0 && r < MD_ROWS) list[r] = threadIdx.x + 256 * u;
      }
      __syncthreads();
      if (WHO == WHO_PAIR && pair >= 0 && list[0] != pair) return;  // (in the pairs' order: another workgroup has the expert)
      x = p.X;
      W += (int64_t)e * (inter ? 2 : 1) * N * K;
      if (W2) W2 += (int64_t)e * N * K;
    }
  }
  auto pair_of = [&](int r) { return LIST || shared_ ? row0 + r : list[r]; };  // the row's place in the results
  auto x_of = [&](int r) {
    const int q = pair_of(min(r, rows - 1));
    return x + (int64_t)(MODE == MD_DOWN || shared_ ? q : LIST ? p.order[q] / p.top : q / p.top) * ldx + (LINES ? 16 : 8) * g;
  };
  auto wa_of = [&](int r) {  // row r of the first group of weight rows, and of the second
    const int n = min(n0 + r, N - 1);
    return W + (int64_t)(MODE == MD_GLU && !plain && inter ? (n >> 4) * 32 + (n & 15) : n) * K;
  };
  auto wb_of = [&](int r) {
    if (MODE == MD_GLU && !plain) return inter ? wa_of(r) + (int64_t)16 * K : W2 + (int64_t)min(n0 + r, N - 1) * K;
    return W + (int64_t)min(n0 + 16 + r, N - 1) * K;
  };
  auto keep = [&](int q, const f32x4& a, const f32x4& b) {
    *reinterpret_cast<f32x4*>(&part[w][0][16 * q + li][4 * g]) = a;
    *reinterpret_cast<f32x4*>(&part[w][1][16 * q + li][4 * g]) = b;
  };
  f32x4 aa[G], ab[G];
  if constexpr (LINES) {
    const int nk = K >> 6, per = (nk + 3) >> 2, s0 = w * per, s1 = min(nk, s0 + per), r8 = lane & 7, c8 = (lane >> 3) * 8;
    const bf16_t* const wa[2] = {wa_of(r8) + c8, wa_of(8 + r8) + c8};
    const bf16_t* const wb[2] = {wb_of(r8) + c8, wb_of(8 + r8) + c8};
    if (LIST || rows <= 16) {
      f32x4 a1[1], b1[1];
      const bf16_t* const xs[1] = {x_of(li)};
      md_products64<1, 4>(wa, wb, xs, s0, s1, a1, b1);
      keep(0, a1[0], b1[0]);
    } else if constexpr (G == 2) {
      const bf16_t* const xs[2] = {x_of(li), x_of(16 + li)};
      md_products64<2, 2>(wa, wb, xs, s0, s1, aa, ab);
      keep(0, aa[0], ab[0]);
      keep(G - 1, aa[G - 1], ab[G - 1]);
    }
  } else {
    const int nk = K >> 5, per = ((nk + 7) >> 3) * 2, s0 = w * per, s1 = min(nk, s0 + per);  // (a wave starts at a line)
    const bf16_t *wa = wa_of(li) + 8 * g, *wb = wb_of(li) + 8 * g;
    if (LIST || rows <= 16) {
      f32x4 a1[1], b1[1];
      const bf16_t* const xs[1] = {x_of(li)};
      md_products<1, 8>(wa, wb, xs, s0, s1, a1, b1);
      keep(0, a1[0], b1[0]);
    } else if constexpr (G == 2) {
      const bf16_t* const xs[2] = {x_of(li), x_of(16 + li)};
      md_products<2, 5>(wa, wb, xs, s0, s1, aa, ab);
      keep(0, aa[0], ab[0]);
      keep(G - 1, aa[G - 1], ab[G - 1]);
    }
  }
  __syncthreads();
  const int c = threadIdx.x & 15;
  for (int r = threadIdx.x >> 4; r < rows; r += 16) {
    float va = 0.f, vb = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      va += part[i][0][r][c];
      vb += part[i][1][r][c];
    }
    const int q = pair_of(r);
    if (shared_ && plain) {
      bf16_t* o = MODE == MD_DOWN ? p.sC + (int64_t)q * N : p.sD + (int64_t)q * p.sldd;
      if (n0 + c < N) o[n0 + c] = f2bf(va);
      if (n0 + 16 + c < N) o[n0 + 16 + c] = f2bf(vb);
      continue;
    }
    const float sw = MODE != MD_DOWN && p.pw && !shared_ ? p.pw[LIST ? p.order[q] : q] : 1.f;
    const int64_t at = (int64_t)q * N + n0 + c;
    if constexpr (MODE == MD_GLU) {
      bf16_t* C = shared_ ? p.sC : (bf16_t*)p.C;
      if (shared_ && !inter) va = bf2f(f2bf(va)), vb = bf2f(f2bf(vb));  // (as its rows are where it runs on its own, in larger steps)
      if (n0 + c < N) C[at] = f2bf(glu_clamped_t(va * sw, vb * sw, shared_ ? p.slimit : p.limit, p.alpha, p.silu));
    } else if constexpr (MODE == MD_GELU) {
      if (n0 + c < N) ((bf16_t*)p.C)[at] = f2bf(gelu_erf(va * sw));
      if (n0 + 16 + c < N) ((bf16_t*)p.C)[at + 16] = f2bf(gelu_erf(vb * sw));
    } else {
      if (n0 + c < N) ((float*)p.C)[at] = va;
      if (n0 + 16 + c < N) ((float*)p.C)[at + 16] = vb;
    }
  }
}

template <int WHO>
static void launch_moe_dec_t(int mode, bool lines, dim3 g, const MoeDecArgs& a, hipStream_t st) {
#define MD_LAUNCH(M_)                                                       \
  do {                                                                      \
    if (lines) moe_dec_kernel<M_, WHO, true><<<g, 256, 0, st>>>(a);        \
    else moe_dec_kernel<M_, WHO, false><<<g, 256, 0, st>>>(a);             \
  } while (0)
  if (mode == MD_GLU) MD_LAUNCH(MD_GLU);
  else if (mode == MD_GELU) MD_LAUNCH(MD_GELU);
  else MD_LAUNCH(MD_DOWN);
#undef MD_LAUNCH
  HIP_CHECK_LAUNCH();
}

// Whether workgroups find their experts' rows themselves (`shared`: the shared expert comes along). What that costs, us: workgroups for pairs
// whose expert another one has (or experts that nobody chose, where pairs are more), 3.9 a thousand; each looks at all pairs; and the
// weights arrive 1 % slower. It saves the grouping launch, and with the shared expert that one's four. Fitted over 4100 random layers (4 - 1024
// experts, 1 - 64 rows, up to 8 pairs an expert), choices at random; over 5200 others 0.76 of the time with a grouping launch, 90 above 1.02, 1.26 at worst
// (8 experts of 1344 x 2304, four pairs 25.9 and 32.7 us).
bool moe_dec_own_rows(int T_, int top, int E, int F, int N, int K, bool glu, bool shared) {
  const double P = (double)T_ * top, n = std::min<double>(E, P), found = E * (1.0 - std::pow(1.0 - (double)top / E, T_));
  const double cols = (F + (glu ? 15 : 31)) / (glu ? 16 : 32) + (N + 31) / 32, weights = 2e-6 * found * F * (K * (glu ? 2.0 : 1.0) + N);
  return 3.9e-3 * (n - found) * cols + 0.002 * P + 0.0095 * weights + 0.7e-6 * P * n * cols < (shared ? 14.6 : 3.3);
}

// mode 0: act [pairs, N] = glu(X W^T, X W2^T) (W2 null: gate and up rows of W [E, 2 N, K] in alternating groups of 16), 1: gelu(X W^T),
// rows of X gathered by token; 2: C = X W^T in fp32, rows of X in the results' order. With a tile list (meta, order, at most maxt tiles):
// results in expert order; without: idx [T, top], results in the pairs' order, `place` [T * top] for modes 0 and 1.
// The shared expert (without a list; s*: null or 0 without one): mode 0: sC [T, sN] = glu of the sN gate and sN up rows of sW (sinter: in
// alternating groups of 16), sD [T, sE] (stride sldd) = the products with sE rows behind them; mode 2: sC [T, N] = sX [T, sK] sW^T.
void launch_moe_dec(int mode, const void* X, int64_t ldx, const void* W, const void* W2, const void* meta, const void* order, void* C,
                    int E, int maxt, int top, int N, int K, float limit, float alpha, const void* pw, int silu, const void* idx,
                    void* place, int T_, const void* sX, const void* sW, void* sC, void* sD, int64_t sldd, int sN, int sK, int sE,
                    int sinter, float slimit, hipStream_t st) {
  const bool list = meta != nullptr;
  if (list ? maxt <= 0 : T_ <= 0) return;
  if (mode < 0 || mode > 2) throw std::runtime_error("moe_dec: mode");
  if (K % 32 || K <= 0 || N <= 0 || ldx % 8 || (((uintptr_t)X | (uintptr_t)W | (uintptr_t)W2) & 15))
    throw std::runtime_error("moe_dec: K % 32, rows of 16-byte alignment");
  if (mode == MD_GLU && !W2 && N % 16) throw std::runtime_error("moe_dec: gate and up in groups of 16 rows");
  MoeDecArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, (const bf16_t*)W2, C, N, K, (const int*)meta, (const int*)order,
               (const float*)pw, E, maxt, top, silu, limit, alpha};
  const int bn = mode == MD_GLU ? 16 : 32;
  if (list) {
    if (maxt > 65535) throw std::runtime_error("moe_dec: too many row tiles");
    if (sW) throw std::runtime_error("moe_dec: no shared expert beside a tile list");
    launch_moe_dec_t<WHO_LIST>(mode, K % 64 == 0, dim3((N + bn - 1) / bn, maxt), a, st);
    return;
  }
  const int64_t P = (int64_t)T_ * top;
  if (P > MD_PAIRS || E <= 0 || E > MD_PAIRS || !idx || (mode != MD_DOWN && !place)) throw std::runtime_error("moe_dec: pairs");
  a.idx = (const int*)idx, a.place = (int*)place, a.P = (int)P, a.xt = (int)P / MD_ROWS;
  int64_t wgs = (std::min<int64_t>(E, P) + a.xt) * ((N + bn - 1) / bn);
  if (sW) {
    if (mode == MD_GELU || sK % 32 || sK <= 0 || sE < 0 || (((uintptr_t)sW | (uintptr_t)sX) & 15) || !sC ||
        (mode == MD_GLU ? sN < 0 || sK != K || (sinter && (sN % 16 || sE)) || (sE && !sD) : sE != 0 || !sX))
      throw std::runtime_error("moe_dec: shared expert");
    a.T = T_, a.sX = (const bf16_t*)sX, a.sW = (const bf16_t*)sW, a.sC = (bf16_t*)sC, a.sD = (bf16_t*)sD, a.sldd = sldd;
    a.sN = sN, a.sK = sK, a.sE = sE, a.sinter = sinter, a.slimit = slimit;
    wgs += (int64_t)((T_ + MD_ROWS - 1) / MD_ROWS) * (((mode == MD_GLU ? sN : N) + bn - 1) / bn + (sE + 31) / 32);
  }
  if (wgs > 0x7fffffff) throw std::runtime_error("moe_dec: too many workgroups");
  const bool lines = K % 64 == 0 && (!sW || sK % 64 == 0);
  if (P < E) launch_moe_dec_t<WHO_PAIR>(mode, lines, dim3((unsigned)wgs), a, st);
  else launch_moe_dec_t<WHO_EXPERT>(mode, lines, dim3((unsigned)wgs), a, st);
}
