// bf16 GEMM of middle sizes: Y[M, N] = epilogue(X[M, K] . W[N, K]^T), K % 64 == 0, on tiles of 32 MT x 32 NT by FOUR waves, each with a
// quarter of the tile (16 MT x 16 NT), K split over the grid where tiles are few. What 256 x 256 tiles (gemm_quad.hip) cannot fill the chip
// with: prompts and mixed steps of some 17 - 4000 rows.
//
// Bound by LDS and the matrix units together: per 64 of k a 128 x 128 tile has its matrix units busy for 0.21 us at 2.4 GHz, LDS for 0.32 (64 KB
// of fragments, 32 KB of loads), 256 x 128 for 0.43 and 0.48, 192 x 192 for 0.48 and 0.48; measured with the chip full 0.44, 0.78 and 0.85 (0.37, 0.65
// and 0.69 with operands of zeros: the rest is the clock under load). Eight waves on a tile of 256 x 128 read 128 KB of fragments a step,
// four read 96: 1.02 us a step there. Both halves of a step's fragments have registers of their own: while one half is multiplied the other is
// read, one barrier a step, behind which the step's buffer is loaded anew, so that a ring of NS has NS - 1 steps on their way. Loads past the
// last step are sent out of the descriptors' range and move nothing.
// The rest of a launch - start, the first step's latency, the epilogue - takes 6 - 9 us of a workgroup alone on its CU (of 5 - 7 of them
// 2 - 3 in the epilogue: 1.7 more at 256 x 128 with stores that stay in the caches, 5 more through fp32 with its activations' code between);
// rings of 48 - 64 KB let two or three workgroups of a CU hide it behind each other.
// us, before and now: 100 rows x 5120 x 2048 15.1 -> 10.7, 512 x 12288 x 4096 73 -> 55, 777 x 2048 x 4096 29 -> 23, 1024 x 4096 x 4096 44 -> 36,
// 1024 x 5120 x 2048 39 -> 28, 1536 x 4096 x 4096 66 -> 48, 1773 x 4096 x 11008 166 -> 139, 2300 x 2048 x 5632 88 -> 55.
#include "common.h"

#include <algorithm>

// Epilogue. The tile goes out through LDS, so that a row leaves in whole lines: as bf16 where the numbers are finished in the registers, as
// fp32 for slabs and where an activation is still to come (its code, unrolled over the accumulators, would not fit the instruction cache).
// 16-byte piece c of row r of an image of CH pieces a row lies at place c ^ (r & four_key(CH)).
constexpr int four_key(int ch) { return (ch & -ch) >= 8 ? 7 : (ch & -ch) - 1; }

template <int MT, int NT>
__device__ __forceinline__ void four_image32(const f32x4 (&acc)[NT][MT], char* smem, int wr, int wc, int li, int g) {
  constexpr int CH = 8 * NT, KEY = four_key(CH);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = wr * MT * 16 + 16 * mt + li;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<f32x4*>(smem + ((r * CH + ((wc * 4 * NT + 4 * nt + g) ^ (r & KEY))) << 4)) = acc[nt][mt];
  }
  __syncthreads();
}

// GLU: groups of 16 columns are gates and their ups in turn
template <int MT, int NT, bool GLU>
__device__ __forceinline__ void four_image16(const f32x4 (&acc)[NT][MT], char* smem, int wr, int wc, int li, int g, int n0, int N,
                                             const bf16_t* __restrict__ bias, int act) {
  constexpr int CH = GLU ? 2 * NT : 4 * NT, KEY = four_key(CH), S = GLU ? 2 : 1;
#pragma unroll
  for (int nt = 0; nt < NT; nt += S) {
    float b[4 * S] = {};
    const int n = n0 + wc * NT * 16 + 16 * nt + 4 * g;
    if (bias && n < N) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        b[i] = bf2f(bias[n + i]);
        if constexpr (GLU) b[4 + i] = bf2f(bias[n + 16 + i]);
      }
    }
    const int c = GLU ? wc * NT + nt + (g >> 1) : wc * 2 * NT + 2 * nt + (g >> 1);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = wr * MT * 16 + 16 * mt + li;
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (GLU) o[i] = f2bf(glu_gate(acc[nt][mt][i] + b[i], act) * (acc[nt + 1][mt][i] + b[4 + i]));
        else o[i] = f2bf(acc[nt][mt][i] + b[i]);
      }
      *reinterpret_cast<u16x4*>(smem + ((r * CH + (c ^ (r & KEY))) << 4) + ((g & 1) << 3)) = o;
    }
  }
  __syncthreads();
}

template <int BM, int BN>
__device__ __forceinline__ void four_store(const char* smem, int m0, int n0, int M, int N, bf16_t* __restrict__ Y, int64_t ldy) {
  constexpr int CH = BN / 8, KEY = four_key(CH);
  bf16_t* const out = Y + (int64_t)m0 * ldy + n0;
#pragma unroll 8
  for (int i = threadIdx.x; i < BM * CH; i += 256) {
    const int r = i / CH, c = i % CH;
    const u16x8 o = *reinterpret_cast<const u16x8*>(smem + ((r * CH + (c ^ (r & KEY))) << 4));
    if (m0 + r < M && n0 + 8 * c < N) __builtin_nontemporal_store(o, reinterpret_cast<u16x8*>(out + (int64_t)r * ldy + 8 * c));
  }
}

template <int BM, int BN, int ACT>
__device__ __forceinline__ void four_store_act(const char* smem, int m0, int n0, int M, int N, bf16_t* __restrict__ Y, int64_t ldy,
                                               const bf16_t* __restrict__ bias) {
  constexpr int CH = BN / 4, KEY = four_key(CH);
  bf16_t* const out = Y + (int64_t)m0 * ldy + n0;
#pragma unroll 2
  for (int i = threadIdx.x; i < BM * CH / 2; i += 256) {
    const int r = i / (CH / 2), c = i % (CH / 2);
    if (m0 + r >= M || n0 + 8 * c >= N) continue;
    f32x4 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) v[h] = *reinterpret_cast<const f32x4*>(smem + ((r * CH + ((2 * c + h) ^ (r & KEY))) << 4));
    u16x8 o, b = {0, 0, 0, 0, 0, 0, 0, 0};
    if (bias) b = *reinterpret_cast<const u16x8*>(bias + n0 + 8 * c);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f2bf(apply_act(v[e >> 2][e & 3] + bf2f(b[e]), ACT));
    *reinterpret_cast<u16x8*>(out + (int64_t)r * ldy + 8 * c) = o;
  }
}

// The query / key / value product: its numbers, rounded as where the rotation is a launch of its own, turned and written to the rows and to
// the paged cache (common.h QkvEpi). Four pieces of a row a thread at a time, their positions and slots, then their angles, then the rest.
template <int BM, int BN>
__device__ __forceinline__ void four_store_qkv(const char* smem, const QkvEpi& e, int m0, int n0, int M, int N, bf16_t* __restrict__ Y,
                                               int64_t ldy) {
  constexpr int CH = BN / 8, KEY = four_key(CH), U = 4;
  const int D = e.D, nq = e.nh * D, nqk = nq + e.nkv * D, rh = e.rot >> 1;
  const bool rope = e.do_rope != 0;
  auto piece = [&](int r, int c) { return *reinterpret_cast<const u16x8*>(smem + ((r * CH + (c ^ (r & KEY))) << 4)); };
#pragma unroll 1
  for (int i0 = threadIdx.x; i0 < BM * CH; i0 += 256 * U) {
    int64_t ps[U], sl[U];
    f32x4 cs[U][2], sn[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = min(m0 + (i0 + 256 * u) / CH, M - 1);
      ps[u] = rope ? e.pos[m] : 0;
      sl[u] = e.kc ? e.slot[m] : -1;
    }
    if (rope) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int n = n0 + (i0 + 256 * u) % CH * 8, d = n % D;
        int a = e.style == 1 ? d >> 1 : (d < rh ? d : d - rh);
        a = n < nqk && d < e.rot ? a : 0;  // (columns that do not turn read an angle that nobody uses)
        const float* cp = e.cos_t + ps[u] * rh + a;
        const float* sp = e.sin_t + ps[u] * rh + a;
        cs[u][0] = *reinterpret_cast<const f32x4*>(cp);
        sn[u][0] = *reinterpret_cast<const f32x4*>(sp);
        if (e.style != 1 && rh >= 8) {
          cs[u][1] = *reinterpret_cast<const f32x4*>(cp + 4);
          sn[u][1] = *reinterpret_cast<const f32x4*>(sp + 4);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + 256 * u, r = i / CH, c = i % CH, m = m0 + r, n = n0 + 8 * c, d = n % D;
      if (i >= BM * CH || m >= M || n >= N) continue;
      u16x8 o = piece(r, c);
      const bool is_v = n >= nqk;
      if (rope && !is_v && d < e.rot) {
        if (e.style == 1) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float x = bf2f(o[2 * k]), y = bf2f(o[2 * k + 1]);
            o[2 * k] = f2bf(x * cs[u][0][k] - y * sn[u][0][k]);
            o[2 * k + 1] = f2bf(y * cs[u][0][k] + x * sn[u][0][k]);
          }
        } else {  // halves of a head turn against each other: both lie in the tile
          const bool lo = d < rh;
          const u16x8 q = piece(r, c + (lo ? rh : -rh) / 8);
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float x = bf2f(o[k]), y = bf2f(q[k]), cv = cs[u][k >> 2][k & 3], sv = sn[u][k >> 2][k & 3];
            o[k] = f2bf(lo ? x * cv - y * sv : x * cv + y * sv);
          }
        }
      }
      *reinterpret_cast<u16x8*>(Y + (int64_t)m * ldy + n) = o;
      if (n >= nq && sl[u] >= 0) {
        const int h = (n - (is_v ? nqk : nq)) / D;
        const int64_t row = ((sl[u] / e.block_size) * e.nkv + h) * (int64_t)e.block_size + sl[u] % e.block_size;
        *reinterpret_cast<u16x8*>((is_v ? e.vc : e.kc) + row * D + d) = o;
      }
    }
  }
}

template <int MT, int NT, int NS>
__global__ __launch_bounds__(256, 1) void gemm_four_kernel(const bf16_t* __restrict__ X, int64_t ldx, const bf16_t* __restrict__ W,
                                                           int64_t ldw, const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                           int64_t ldy, float* __restrict__ part, int M, int N, int K, int act, int glu,
                                                           int split, int group_m, int* __restrict__ cnt, QkvEpi qe) {
  constexpr int BM = 32 * MT, BN = 32 * NT, XB = BM * 128, STAGE = (BM + BN) * 128, LOADS = MT + NT;
  static_assert(NS >= 2 && NS * STAGE <= 160 * 1024 && (NS - 1) * LOADS <= 63, "ring");
  static_assert(BM * BN * 4 <= NS * STAGE, "the epilogue's image lies in the ring");
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4, wr = w >> 1, wc = w & 1;
  const int ntn = (N + BN - 1) / BN, ntm = (M + BM - 1) / BM, tiles = ntm * ntn;
  const int id = xcd_remap(blockIdx.x, tiles * split);
  const int zk = id / tiles, tile = id - zk * tiles;
  const int grp = tile / (group_m * ntn), gidx = tile - grp * (group_m * ntn);
  const int gm = min(group_m, ntm - grp * group_m);
  const int m0 = (grp * group_m + gidx % gm) * BM, n0 = (gidx / gm) * BN;
  const int nk = K >> 6, per = (nk + split - 1) / split, t0 = zk * per, t1 = min(nk, t0 + per);
  // rows past the last one lie outside the descriptors and read as zeros
  const uint64_t xbytes = (uint64_t)(M - m0) * (uint64_t)ldx * 2, wbytes = (uint64_t)(N - n0) * (uint64_t)ldw * 2;
  const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(X) + (int64_t)m0 * ldx * 2), (short)0,
                                                    (int)(xbytes > 0x7FFFFFF0ull ? 0x7FFFFFF0u : (uint32_t)xbytes), 0x00020000);
  const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(W) + (int64_t)n0 * ldw * 2), (short)0,
                                                    (int)(wbytes > 0x7FFFFFF0ull ? 0x7FFFFFF0u : (uint32_t)wbytes), 0x00020000);
  uint32_t vx[MT], vw[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row = (i * 4 + w) * 8 + (lane >> 3);
    vx[i] = (uint32_t)row * (uint32_t)(ldx * 2) + (uint32_t)(((lane & 7) ^ (row & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int row = (i * 4 + w) * 8 + (lane >> 3);
    vw[i] = (uint32_t)row * (uint32_t)(ldw * 2) + (uint32_t)(((lane & 7) ^ (row & 7)) << 4);
  }
  // load I_ (eight rows, 1 KB) of k-step T_ into the buffer at B_; OUT_: past the last step, as an offset that no descriptor reaches
#define F_LOAD(I_, T_, B_, OUT_)                                                                                                     \
  do {                                                                                                                               \
    if ((I_) < MT)                                                                                                                   \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (LDS_AS void*)(smem + (B_) + ((I_) * 4 + w) * 1024), 16,                            \
                                               (uint32_t)(vx[(I_) < MT ? (I_) : 0] | (OUT_)), (uint32_t)((T_) * 128), 0, 0);          \
    else                                                                                                                             \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (LDS_AS void*)(smem + (B_) + XB + (((I_) - MT) * 4 + w) * 1024), 16,                \
                                               (uint32_t)(vw[(I_) < MT ? 0 : (I_) - MT] | (OUT_)), (uint32_t)((T_) * 128), 0, 0);     \
  } while (0)
  const int xo = (wr * MT * 16 + li) * 128 + ((g ^ (li & 7)) << 4);
  const int wo = XB + (wc * NT * 16 + li) * 128 + ((g ^ (li & 7)) << 4);
#define F_READ(P_, T_) (*reinterpret_cast<const s16x8*>(smem + (P_) + (T_) * 2048))
  f32x4 acc[NT][MT];  // a lane: of row 16 mt + li, the four columns 16 nt + 4 g
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  s16x8 x0[MT], w0[NT], x1[MT], w1[NT];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const uint32_t out = t0 + s < t1 ? 0u : 0x80000000u;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) F_LOAD(i, t0 + s, s * STAGE, out);
  }
  constexpr int V0 = (NS - 1) * LOADS, V1 = (NS - 2) * LOADS;
  __builtin_amdgcn_s_waitcnt((V0 & 15) | (7 << 4) | (15 << 8) | ((V0 >> 4) << 14));  // the first step has landed
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < NT; ++q) w0[q] = F_READ(wo, q);
#pragma unroll
  for (int q = 0; q < MT; ++q) x0[q] = F_READ(xo, q);
  // in place by the instruction's own operands: left to itself the compiler moves every accumulator between the register files and back
#define F_MFMA(X_, W_, MT_, NT_)                                                                                                     \
  do {                                                                                                                               \
    if constexpr (MT * NT >= 32) asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[NT_][MT_]) : "v"(W_[NT_]), "v"(X_[MT_]));  \
    else asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[NT_][MT_]) : "v"(W_[NT_]), "v"(X_[MT_]));                          \
  } while (0)
  constexpr int G = MT * NT, NR = MT + NT, RP = (2 * NR + G - 1) / G;  // products and fragment reads of half a step; reads per two products
  constexpr int LP = (2 * LOADS + G - 1) / G;                          // loads per two products
  int cx = 0;
#pragma unroll 1
  for (int t = t0; t < t1; ++t) {
    const int nx = cx == (NS - 1) * STAGE ? 0 : cx + STAGE;
    const int xa = cx + (xo ^ 64), wa = cx + (wo ^ 64), xb = nx + xo, wb = nx + wo;
    const uint32_t out = t + NS < t1 ? 0u : 0x80000000u;
#pragma unroll
    for (int q = 0; q < (G + 1) / 2; ++q) {
#pragma unroll
      for (int r = q * RP; r < (q + 1) * RP && r < NR; ++r) {
        if (r < NT) w1[r < NT ? r : 0] = F_READ(wa, r);
        else x1[r < NT ? 0 : r - NT] = F_READ(xa, r - NT);
      }
#pragma unroll
      for (int p = 2 * q; p < 2 * q + 2 && p < G; ++p)
        F_MFMA(x0, w0, p / NT, p % NT);
      __builtin_amdgcn_sched_barrier(0);
    }
    // this step is read, this wave's part of the next has landed
    __builtin_amdgcn_s_waitcnt((V1 & 15) | (7 << 4) | ((V1 >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < (G + 1) / 2; ++q) {
#pragma unroll
      for (int r = q * RP; r < (q + 1) * RP && r < NR; ++r) {
        if (r < NT) w0[r < NT ? r : 0] = F_READ(wb, r);
        else x0[r < NT ? 0 : r - NT] = F_READ(xb, r - NT);
      }
#pragma unroll
      for (int l = q * LP; l < (q + 1) * LP && l < LOADS; ++l) F_LOAD(l, t + NS, cx, out);
#pragma unroll
      for (int p = 2 * q; p < 2 * q + 2 && p < G; ++p)
        F_MFMA(x1, w1, p / NT, p % NT);
      __builtin_amdgcn_sched_barrier(0);
    }
    cx = nx;
  }
#undef F_MFMA
#undef F_READ
#undef F_LOAD
  __builtin_amdgcn_s_waitcnt(0x0070);                  // no load of this wave is on its way into LDS any more,
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // and the last products are written, which the compiler does not see
  __builtin_amdgcn_sched_barrier(0);
  if (cnt) {  // split-K slices combine in this launch; the tile's last arriver runs the epilogue
    if (!splitk_combine<NT, MT>(acc, part, cnt, tile, split, zk, w, 4, lane, reinterpret_cast<int*>(smem))) return;
    part = nullptr;
  }
  __builtin_amdgcn_s_barrier();  // every wave is done with the ring
  __builtin_amdgcn_sched_barrier(0);
  if (part) {
    four_image32<MT, NT>(acc, smem, wr, wc, li, g);
    constexpr int CH = BN / 4, KEY = four_key(CH);
    float* const out = part + (int64_t)zk * M * N + (int64_t)m0 * N + n0;
#pragma unroll 8
    for (int i = threadIdx.x; i < BM * CH; i += 256) {
      const int r = i / CH, c = i % CH;
      const f32x4 v = *reinterpret_cast<const f32x4*>(smem + ((r * CH + (c ^ (r & KEY))) << 4));
      if (m0 + r < M && n0 + 4 * c < N) *reinterpret_cast<f32x4*>(out + (int64_t)r * N + 4 * c) = v;
    }
    return;
  }
  if (qe.D) {
    four_image16<MT, NT, false>(acc, smem, wr, wc, li, g, n0, N, bias, 0);
    four_store_qkv<BM, BN>(smem, qe, m0, n0, M, N, Y, ldy);
    return;
  }
  if constexpr (NT % 2 == 0) {
    if (glu) {
      four_image16<MT, NT, true>(acc, smem, wr, wc, li, g, n0, N, bias, act);
      four_store<BM, BN / 2>(smem, m0, n0 / 2, M, N / 2, Y, ldy);
      return;
    }
  }
  if (act == ACT_NONE) {
    four_image16<MT, NT, false>(acc, smem, wr, wc, li, g, n0, N, bias, 0);
    four_store<BM, BN>(smem, m0, n0, M, N, Y, ldy);
    return;
  }
  four_image32<MT, NT>(acc, smem, wr, wc, li, g);
  if (act == ACT_GELU_TANH) four_store_act<BM, BN, ACT_GELU_TANH>(smem, m0, n0, M, N, Y, ldy, bias);
  else if (act == ACT_GELU) four_store_act<BM, BN, ACT_GELU>(smem, m0, n0, M, N, Y, ldy, bias);
  else if (act == ACT_RELU) four_store_act<BM, BN, ACT_RELU>(smem, m0, n0, M, N, Y, ldy, bias);
  else four_store_act<BM, BN, ACT_RELU2>(smem, m0, n0, M, N, Y, ldy, bias);
}

// code, MT, NT, ring: rings of 48 - 80 KB leave room for a second or third workgroup on a CU, the others take it whole
#define FOUR_TILES(F)                                                                                                              \
  F(0, 2, 2, 3) F(1, 1, 2, 5) F(2, 4, 2, 3) F(3, 4, 4, 2) F(4, 4, 4, 4) F(5, 6, 4, 4) F(6, 4, 6, 4) F(7, 8, 4, 3) F(8, 2, 1, 5) \
  F(9, 6, 6, 3) F(10, 2, 4, 3) F(11, 4, 2, 6) F(12, 2, 4, 6) F(13, 2, 2, 8)

bool gemm_four_dims(int code, int* bm, int* bn) {
#define F(C_, MT_, NT_, NS_) \
  if (code == C_) { *bm = 32 * MT_; *bn = 32 * NT_; return true; }
  FOUR_TILES(F)
#undef F
  return false;
}

// any of the tiles takes these operands
bool gemm_four_ok(int N, int K, int64_t ldx, int64_t ldw, const void* Y, int64_t ldy, bool glu) {
  return K % 64 == 0 && K > 0 && N % (glu ? 32 : 8) == 0 && ldx % 8 == 0 && ldw % 8 == 0 && std::max(ldx, ldw) < (1 << 22) - 64 &&
         ((uintptr_t)Y & 15) == 0 && ldy % 8 == 0;
}

void launch_gemm_four(int code, const bf16_t* X, int64_t ldx, const bf16_t* W, int64_t ldw, const bf16_t* bias, bf16_t* Y, int64_t ldy, float* part,
                      int M, int N, int K, int act, int glu, int split, int group_m, hipStream_t st, int* cnt, const QkvEpi* qe) {
  int bm, bn;
  if (!gemm_four_ok(N, K, ldx, ldw, Y, ldy, glu != 0) || !gemm_four_dims(code, &bm, &bn) || (glu && bn % 64)) throw std::runtime_error("gemm_four: operands or tile");
  const unsigned nwg = (unsigned)(((M + bm - 1) / bm) * ((N + bn - 1) / bn) * split);
  const QkvEpi qv = qe ? *qe : QkvEpi{};
#define F(C_, MT_, NT_, NS_)                                                                                                              \
  case C_:                                                                                                                                \
    gemm_four_kernel<MT_, NT_, NS_><<<nwg, 256, 0, st>>>(X, ldx, W, ldw, bias, Y, ldy, part, M, N, K, act, glu, split, group_m, cnt, qv); \
    break;
  switch (code) { FOUR_TILES(F) }
#undef F
  HIP_CHECK_LAUNCH();
}
