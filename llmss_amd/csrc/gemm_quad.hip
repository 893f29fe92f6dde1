// Prompt GEMM (bf16, K % 64 == 0): Y[M, N] = epilogue(X[M, K] . W[N, K]^T) on 256 x 256 tiles by FOUR waves, a wave per SIMD with a
// 128 x 128 part of the tile.
//
// Bound by the matrix units at the clock that the chip holds under them: over 8192 x 12288 x 4096 it is 1.43 - 1.93 GHz (GRBM_GUI_ACTIVE
// over the launch's time; 2.4 nominal) and the matrix units are busy for 67 - 73 % of the cycles (SQ_VALU_MFMA_BUSY_CYCLES). With loads
// and epilogue taken out, 64 of k take a wave of 256 tiles 1.27 us (0.85 us of issue at 2.4 GHz), and 1.5 us as it stands. Per 64
// of k a wave reads (128 + 128) x 64 for 128 products, half of what eight waves read together, and the reads are free behind them. What
// costs is the loads and the epilogue:
// - a step's loads are issued 1.5 (X) and 1 (W) steps before the barrier that waits for them, by count. With a step's distance of less than
//   one (two buffers) it took 1.63 - 1.84 us; a ring of four 32-k buffers, with more distance but rows of 64 bytes, 1.6 - 1.75 us.
// - the start of a tile and its end, 8.5 us of 53 at K = 2048 while each tile was a workgroup: 42 us a tile with stores of 64 bytes a row straight
//   from the accumulators, 20 us through LDS with the activations' code unrolled (36 KB of it), 6 - 8 us through LDS as written at the end. So
//   a workgroup now takes every 256th tile (RING): the ring of loads runs on into the next tile while the last steps of this one are
//   multiplied, and the tile leaves straight from the accumulators in whole lines, without LDS (quad_store): 5.7 us a tile. The clock gives a
//   part back: matrix units that are busy for more of the time run slower. us: 8192 x 10240 x 2048 248 -> 241, x 9472 243 -> 233, SwiGLU
//   8192 x 11264 x 2048 297 -> 280, x 4096 105 -> 100, 8192 x 8192 x 768 97 -> 88, SwiGLU 8192 x 22016 x 4096 1047 -> 1017, 8192 x 5120 x 2048 143 -> 138;
//   one tile a CU is as before (8192 x 2048 x 4096 100). Prompts of Babotar 5831 -> 5694, Fizelix 6963 -> 6823, Nolavik 5024 -> 4919.
//   Products with an activation but no gate, whose code does not fit beside so many accumulators, and the query / key / value product with its
//   rotation keep the way through LDS.
// Against the ping-pong kernel of 8 waves (weights not in the caches, us): 8192 x 12288 x 4096 794 -> 715, 8192 x 4096 x 4096 232 -> 206,
// 8192 x 4096 x 11008 540 -> 530, 8192 x 11264 x 2048 379 -> 330; SwiGLU 8192 x 22016 x 4096 1237 (1195 TFLOP/s).
//
// GRP: grouped expert products over moe.hip's list of 256-row tiles, as in the ping-pong kernel: 1 - rows of X gathered through
// order[] / top, activation or gating in the epilogue; 2 - rows in expert order, fp32 output; 3 - as 1 with GLU over two
// matrices, gate and up, the products scaled by the pair's weight first. GLU: W's rows are gate and up in alternating groups of 16.
#include "gemm_quad.h"

#include <algorithm>
#include <type_traits>

// The wave's 128 x 128 part of a finished tile (GRP: every other sixteen rows from m0 on; half: four of them), straight from the accumulators.
// A lane holds, of row MS mt + li, sixteen bytes of neighbouring
// columns (two tiles of eight: GLU, four gates and their four ups twice; fp32: one tile of four) - 64 bytes a row and instruction, and stores of
// half lines take four times as long. So two such pieces change hands between lanes li and li ^ 8 (a rotation by eight within the row of
// sixteen lanes): one instruction then writes rows 0 .. 7 of the sixteen in whole lines, another rows 8 .. 15.
// Rows and columns past the last lie outside the descriptor, so that no branch stands between the stores. (gemm_quad_ok: the rows that a wave
// reaches over, 240 where they alternate by sixteens and else 128, fit a descriptor of 31 bits.)
// PAST: past the caches, as bf16 results (65536 pairs x 768 390 -> 367 us with all of their product) and fp32 sums that these would not hold until they
// are read: of 32768 pairs x 2048 (K = 768) 152 -> 131 us. Up to 128 MB are in them when the combining launch reads them (launch_gemm_quad).
template <int GRP, int GLU, int MS, bool PAST>
__device__ __forceinline__ void quad_store(const f32x4 (&acc)[8][8], const PpGroup& gr, const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                           int64_t ldy, int m0, int n0, int M, int N, int li, int g, const float (&sw)[8], bool half) {
  constexpr int ES = GRP == 2 ? 4 : 2, COLS = GRP == 2 ? 4 : GLU ? 1 : 2, RUN = GRP == 2 ? 32 : 64;  // runs of a line
  const int nout = GLU ? N / 2 : N, o0 = GLU ? n0 / 2 : n0, up = li >> 3;
  const uint32_t pitch = (uint32_t)ldy * ES;
  const GluForm glu(gr.limit, gr.alpha, gr.silu);
  const auto ry = uniform_rsrc((GRP == 2 ? reinterpret_cast<char*>(gr.Yf) : reinterpret_cast<char*>(Y)) + (int64_t)m0 * ldy * ES,
                               (int64_t)max(min(M - m0, 7 * MS + 16), 0) * pitch);
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    float bs[2][GLU ? 16 : 8] = {};
    if (GRP != 2 && bias) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          // (GLU: bias lies as W's rows, gates and ups in groups of 16)
          const int n = GLU ? n0 + 64 * h + 32 * (g >> 1) + 8 * (g & 1) + i : n0 + 64 * c + 32 * h + 8 * g + i;
          bs[h][i] = n < N ? bf2f(bias[n]) : 0.f;
          if constexpr (GLU) bs[h][8 + i] = n < N ? bf2f(bias[n + 16]) : 0.f;
        }
    }
    const int n = o0 + RUN * c + RUN / 2 * up + RUN / 8 * g;
    const uint32_t at = (uint32_t)(li & 7) * pitch + (uint32_t)n * ES;
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      if (GRP != 0 && mt == 4 && half) break;
      u32x4 a, b;
      if constexpr (GRP == 2) {
        a = __builtin_bit_cast(u32x4, acc[2 * c][mt]), b = __builtin_bit_cast(u32x4, acc[2 * c + 1][mt]);
      } else {
        u16x8 o[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if constexpr (GLU) {
              const int t = 4 * h + 2 * (i >> 2);
              const float gv = acc[t][mt][i & 3], uv = acc[t + 1][mt][i & 3];
              if constexpr (GRP == 3) o[h][i] = f2bf(glu(gv * sw[mt], uv * sw[mt]));
              else o[h][i] = f2bf((GLU == 2 ? gelu_gate_by(gv + bs[h][i]) : silu_gate_by(gv + bs[h][i])) * (uv + bs[h][8 + i]));
            } else {
              o[h][i] = f2bf(acc[4 * c + 2 * h + (i >> 2)][mt][i & 3] + bs[h][i]);
            }
          }
        a = __builtin_bit_cast(u32x4, o[0]), b = __builtin_bit_cast(u32x4, o[1]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t x = a[i], y = b[i];
        a[i] = __builtin_amdgcn_update_dpp(x, y, 0x128, 0xf, 0xc, false);  // lanes 8 .. 15: of b, from li - 8
        b[i] = __builtin_amdgcn_update_dpp(y, x, 0x128, 0xf, 0x3, false);  // lanes 0 .. 7: of a, from li + 8
      }
      const uint32_t ra = n < nout ? at + (uint32_t)(MS * mt) * pitch : ~0u, rb = n < nout ? at + (uint32_t)(MS * mt + 8) * pitch : ~0u;
      __builtin_amdgcn_raw_buffer_store_b128(a, ry, ra, 0, PAST ? 2 : 0);
      __builtin_amdgcn_raw_buffer_store_b128(b, ry, rb, 0, PAST ? 2 : 0);
    }
  }
}

// GLU 1: SiLU gates, 2: the tanh form of GELU, 8192 x 11264 x 2048 with its gate 323 us (the product alone 306, with a launch of its own for the
// gate 356; 64 rows 15.5 and 17.3, one row 11.2 and 13.0)
// QKV: the query / key / value product, its rows turned (neighbouring pairs, or not at all) and its keys and values written to the paged cache on
// the way out (common.h QkvEpi). The wave's 128 columns go out as one image of bf16 - the numbers are rounded before they are turned, as where
// the rotation is a launch of its own - whose 16 pieces of a row are one lane's columns throughout; where a row lies in the cache is
// looked up once a row and kept in the ring's fifth buffer.
// Against the product and a rotation of its own, which reads and writes all of it again (us): 8192 x 12288 x 4096 676 -> 621, 3999 rows 343 ->
// 315; 8192 x 4800 x 1600 without a rotation 159 -> 140.
template <int GRP, int GLU, bool QKV = false, bool RING = false, bool PAST = true>
__global__ __launch_bounds__(256, 1) void gemm_quad_kernel(const bf16_t* __restrict__ X, int64_t ldx,
                                                           const bf16_t* __restrict__ W, int64_t ldw,
                                                           const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y,
                                                           int64_t ldy, int M, int N, int K, int act, int group_m, PpGroup gr, QkvEpi qe) {
  static_assert(!QKV || (GRP == 0 && GLU == 0), "QKV: plain products");
  // a ring of five buffers, each 64 of k (128 bytes, a line) of 256 rows: X of step 0, W of step 0, X of step 1, ...
  constexpr int BUF = 32768, NB = 5, QA = 6;
  constexpr bool GATHER = GRP == 1 || GRP == 3, HALF = RING && GRP != 0;
  __shared__ __attribute__((aligned(16))) char smem[NB * BUF];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wr = w >> 1, wc = w & 1;
  const int ntn = (N + 255) / 256, ntm = (M + 255) / 256;
  const int tiles = GRP != 0 ? __builtin_amdgcn_readfirstlane(gr.meta[0]) * ntn : ntn * ntm;
  if ((int)blockIdx.x >= tiles) return;
  const int nk = K >> 6;
  if (GRP == 3 && (w & 2)) W = gr.Wu;
  // Expert lists: first the tiles of more than 128 rows, tall of them, round by round, then the half tiles, whose upper products are left out.
  // Workgroups that have one round less begin with those, two each, before the others get any. 32 experts of 2048 x 768, us: 1024 pairs each by
  // chance, a rest of some rows for every other, first product 228 -> 201 (170 without rests: half tiles read weights that have left the caches,
  // a step a microsecond), second 156 -> 130; 320 each 110 -> 91 and 55 -> 57; 16 of 1024 x 512 by about 900, 68 -> 45 and 43 -> 31.
  const int G = gridDim.x, tall = HALF ? __builtin_amdgcn_readfirstlane(gr.meta[2 + gr.E + 2 * gr.maxt]) * ntn : tiles;
  const int over = tall % G;  // workgroups that have a round more
  const int rounds = tall / G + ((int)blockIdx.x < over);
  // number i of this workgroup's tiles, or -1
  auto tile_no = [&](int i) {
    const int b = (int)blockIdx.x;
    if (!RING) return i ? -1 : xcd_remap(b, tiles);
    if (i < rounds) return xcd_remap(b + i * G, tall);
    const int k = i - rounds, early = b >= over ? 2 : 0;
    const int t = tall + (k < early ? b - over + k * (G - over) : 2 * (G - over) + b + (k - early) * G);
    return t < tiles ? t : -1;
  };
  // tile id: its first row and column, the rows that there are, and where its operands lie (bytes that exist from there on)
  struct Tile {
    int m0, n0, M;
    const char *x, *w;
    uint32_t xb, wb;
  };
  auto place = [&](int id) {
    Tile t;
    const bf16_t* wt = W;
    t.M = M;
    if constexpr (GRP != 0) {
      const int ty = id / ntn;
      const int e = __builtin_amdgcn_readfirstlane(gr.meta[1 + (gr.E + 1) + ty]);
      t.n0 = (id - ty * ntn) * 256;
      t.m0 = __builtin_amdgcn_readfirstlane(gr.meta[1 + (gr.E + 1) + gr.maxt + ty]);
      t.M = __builtin_amdgcn_readfirstlane(gr.meta[1 + e + 1]);
      wt += (int64_t)e * gr.sB;
    } else {
      const int grp = id / (group_m * ntn), gidx = id - grp * (group_m * ntn);
      const int gm = min(group_m, ntm - grp * group_m);
      t.m0 = (grp * group_m + gidx % gm) * 256, t.n0 = (gidx / gm) * 256;
    }
    const uint64_t xb = GATHER ? ~0ull : (uint64_t)(t.M - t.m0) * (uint64_t)ldx * 2;
    // (rows 16 .. 31 of every 32 of a tile are up rows: a load takes eight rows, so a wave's loads are all of one matrix)
    const uint64_t wb = (uint64_t)(GRP == 3 ? (N - t.n0) / 2 : N - t.n0) * (uint64_t)ldw * 2;
    t.x = reinterpret_cast<const char*>(X) + (GATHER ? 0 : (int64_t)t.m0 * ldx * 2);
    t.w = reinterpret_cast<const char*>(wt) + (int64_t)(GRP == 3 ? t.n0 / 2 : t.n0) * ldw * 2;
    t.xb = xb > 0xFFFFFFF0ull ? 0xFFFFFFF0u : (uint32_t)xb;
    t.wb = wb > 0xFFFFFFF0ull ? 0xFFFFFFF0u : (uint32_t)wb;
    return t;
  };
  int at = 0, ahead = RING ? tile_no(1) : -1;
  const int first = tile_no(0);
  if (first < 0) return;
  Tile cur = place(first), next = cur;
  if constexpr (RING) {
    if (ahead >= 0) next = place(ahead);
    else next.xb = next.wb = 0;  // (nothing is in its range)
  }
  // chunk c of row r lies at place c ^ key(r) of the row: the eight rows that a fragment read's eight lanes take fall on eight
  // different 16-byte columns of the banks
  auto xkey = [](int r) { return r & 7; };
  // (W's rows as they come, or so that a lane gets eight neighbouring columns in two tiles, below)
  constexpr bool PLAIN = RING ? GRP == 2 : GLU != 0;
  auto wkey = [](int r) { return PLAIN ? r & 7 : (r & 3) | ((r >> 3) & 1) << 2; };
  uint32_t vx[8], vw[8], vn[8];
  // rows of X that a lane loads (GATHER: by pair), and what its pairs weigh
  auto pair_of = [&](const Tile& t, int i) { return GATHER ? gr.order[min(t.m0 + (i * 4 + w) * 8 + (lane >> 3), t.M - 1)] : 0; };
  auto offset_of = [&](int pair, int i) {
    const int row = (i * 4 + w) * 8 + (lane >> 3);
    return (uint32_t)(GATHER ? pair / gr.top : row) * (uint32_t)(ldx * 2) + (uint32_t)(((lane & 7) ^ xkey(row)) << 4);
  };
  auto weight_of = [&](const Tile& t, int mt) { return gr.pw ? gr.pw[gr.order[min(t.m0 + 32 * mt + 16 * wr + li, t.M - 1)]] : 1.f; };
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = (i * 4 + w) * 8 + (lane >> 3);
    vx[i] = offset_of(pair_of(cur, i), i);
    if constexpr (RING && GATHER) vn[i] = offset_of(pair_of(next, i), i);
    const int wrw = GRP == 3 ? (row >> 5) * 16 + (row & 15) : row;
    vw[i] = (uint32_t)wrw * (uint32_t)(ldw * 2) + (uint32_t)(((lane & 7) ^ wkey(row)) << 4);
  }
  // eight rows (1 KB) of step T_ of X or W into buffer B_
#define Q_RSRC(P_, B_) __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(P_), (short)0, (int)(B_), 0x00020000)
#define Q_LOAD(R_, V_, I_, T_, B_)                                                                                    \
  __builtin_amdgcn_raw_ptr_buffer_load_lds(R_, (LDS_AS void*)(smem + (B_) + ((I_) * 4 + w) * 1024), 16, (uint32_t)(V_), (uint32_t)((T_) * 128), 0, 0)
  const int wrow = PLAIN ? li : (GLU ? 32 * (li >> 3) + 8 * ((li >> 2) & 1) + (li & 3) : 8 * (li >> 2) + (li & 3));
  // (HALF: the waves' rows alternate by sixteens, so that a tile of up to 128 rows is the first half of both waves' products)
  constexpr int XT = HALF ? 4096 : 2048;
  const int xo = (wr * (HALF ? 16 : 128) + li) * 128 + ((g ^ xkey(li)) << 4);
  const int wo = (wc * 128 + wrow) * 128 + ((g ^ wkey(wrow)) << 4);
#define Q_X(P_, T_) (*reinterpret_cast<const s16x8*>(smem + (P_) + (T_) * XT))
#define Q_W(P_, T_)                                \
  (*reinterpret_cast<const s16x8*>(smem + (P_) + (PLAIN ? (T_) * 2048                                                        \
                                                  : GLU ? ((T_) >> 2) * 8192 + (((T_) >> 1) & 1) * 512 + ((T_) & 1) * 2048  \
                                                        : ((T_) >> 1) * 4096 + ((T_) & 1) * 512)))
  f32x4 acc[8][8];  // [W tile][X tile]
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  s16x8 w0[8], x0[8], w1[8], x1[8];
  // In place by the instruction's own operands: left to itself the compiler, with every accumulation register taken, rotates the
  // accumulators through the file by 272 moves per 64 of k. A quarter of them lives in the vector file, so that both have room.
#define Q_MFMA(W_, X_, NT_, MT_)                                                                                          \
  do {                                                                                                                    \
    if ((NT_) < QA)                                                                                                       \
      asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[NT_][MT_]) : "v"(W_[NT_]), "v"(X_[MT_]));                  \
    else                                                                                                                  \
      asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[NT_][MT_]) : "v"(W_[NT_]), "v"(X_[MT_]));                  \
  } while (0)
  // The products of W tiles NT_ and NT_ + 1 with X tiles 4 .. 7, which half tiles pass over. The branch stands inside, for the compiler moves and
  // spills accumulators around one that it sees; one for eight products costs whole tiles 2 % (one for four 4 %).
#define Q_UPPER8(C_, W_, X_, NT_)                                                                                         \
  asm("s_cmp_lg_u32 %14, 0\n\ts_cbranch_scc0 1f\n\t"                                                                    \
      "v_mfma_f32_16x16x32_bf16 %0, %8, %10, %0\n\tv_mfma_f32_16x16x32_bf16 %1, %8, %11, %1\n\t"                        \
      "v_mfma_f32_16x16x32_bf16 %2, %8, %12, %2\n\tv_mfma_f32_16x16x32_bf16 %3, %8, %13, %3\n\t"                        \
      "v_mfma_f32_16x16x32_bf16 %4, %9, %10, %4\n\tv_mfma_f32_16x16x32_bf16 %5, %9, %11, %5\n\t"                        \
      "v_mfma_f32_16x16x32_bf16 %6, %9, %12, %6\n\tv_mfma_f32_16x16x32_bf16 %7, %9, %13, %7\n1:"                        \
      : "+" C_(acc[NT_][4]), "+" C_(acc[NT_][5]), "+" C_(acc[NT_][6]), "+" C_(acc[NT_][7]), "+" C_(acc[NT_ + 1][4]),      \
        "+" C_(acc[NT_ + 1][5]), "+" C_(acc[NT_ + 1][6]), "+" C_(acc[NT_ + 1][7])                                         \
      : "v"(W_[NT_]), "v"(W_[NT_ + 1]), "v"(X_[4]), "v"(X_[5]), "v"(X_[6]), "v"(X_[7]), "s"(full)                         \
      : "scc")
  // A step's 64 products over its 16 places, four each (HALF: tiles 4 .. 7 of two W tiles in every fourth place).
#define Q_FOUR(W_, X_, Q_)                                                                                    \
  do {                                                                                                        \
    const int nt = (Q_) >> 1;                                                                                 \
    if (HALF && ((Q_) & 3) == 3) {                                                                            \
      if (nt < QA) Q_UPPER8("a", W_, X_, nt - 1);                                                             \
      else Q_UPPER8("v", W_, X_, nt - 1);                                                                     \
    } else if (!HALF || ((Q_) & 3) != 2) {                                                                    \
      const int n1 = HALF ? nt + ((Q_) & 1) : nt, m1 = HALF ? 0 : ((Q_) & 1) * 4;                             \
      _Pragma("unroll") for (int e = 0; e < 4; ++e) Q_MFMA(W_, X_, n1, m1 + e);                               \
    }                                                                                                         \
  } while (0)
  {
    const auto rx = Q_RSRC(cur.x, cur.xb), rw = Q_RSRC(cur.w, cur.wb);
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      const int t = min(l >> 1, nk - 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (l & 1) Q_LOAD(rw, vw[i], i, t, l * BUF);
        else Q_LOAD(rx, vx[i], i, t, l * BUF);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x4F78);  // vmcnt(24): the first step has landed
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    w0[q] = Q_W(BUF + wo, q);
    x0[q] = Q_X(xo, q);
  }
  int cx = 0;  // buffer of this step's X; its W lies in the next one
#pragma unroll 1
  for (;;) {
    // One copy of the body: with separate last steps the compiler moves every accumulator between register files. The last steps load the
    // next tile's first ones (RING; or the last one again), and the very last reads its fragments (or some that nobody uses).
    // (the builtin is taken out as one of a uniform value, which then lies in a vector register)
    int full = 1;
    if constexpr (HALF) asm("s_nop 4\n\tv_readfirstlane_b32 %0, %1\n\ts_nop 4" : "=s"(full) : "v"((int)(cur.M - cur.m0 > 128)));
#pragma unroll 1
    for (int t = 0; t < nk; ++t) {
      const int cw = cx == 4 * BUF ? 0 : cx + BUF;
      const int nx = cw == 4 * BUF ? 0 : cw + BUF;
      const int nw = nx == 4 * BUF ? 0 : nx + BUF;
      const int xa = cx + (xo ^ 64), wa = cw + (wo ^ 64), xb = nx + xo, wb = nw + wo;
      const bool wn = RING && t + 2 >= nk, xn = RING && t + 3 >= nk;
      const int tw = RING ? t + 2 - (wn ? nk : 0) : min(t + 2, nk - 1), tx = RING ? t + 3 - (xn ? nk : 0) : min(t + 3, nk - 1);
      const auto rx = Q_RSRC(xn ? next.x : cur.x, xn ? next.xb : cur.xb), rw = Q_RSRC(wn ? next.w : cur.w, wn ? next.wb : cur.wb);
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        if (q < 8) {
          w1[q] = Q_W(wa, q);
          x1[q] = Q_X(xa, q);
        }
        Q_FOUR(w0, x0, q);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_waitcnt(0x0078);  // vmcnt(8) lgkmcnt(0): this step is read, this wave's part of the next has landed
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        if (q < 8) {
          w0[q] = Q_W(wb, q);
          x0[q] = Q_X(xb, q);
          Q_LOAD(rw, vw[q], q, tw, cx);
        } else {
          Q_LOAD(rx, RING && GATHER && xn ? vn[q - 8] : vx[q - 8], q - 8, tx, cw);
        }
        Q_FOUR(w1, x1, q);
        __builtin_amdgcn_sched_barrier(0);
      }
      cx = nx;
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products are written, which the compiler does not see
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!RING) {
      break;
    } else {
      // (what the tile after the next needs of the lists is asked for before the stores, behind which it would wait)
      Tile then = next;
      const int after = ahead < 0 ? -1 : tile_no(++at + 1);
      if (after >= 0) then = place(after);
      else then.xb = then.wb = 0;
      int pairs[8];
      float sw[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (GATHER) pairs[i] = pair_of(then, i);
        if constexpr (GRP == 3) sw[i] = weight_of(cur, i);
      }
      __builtin_amdgcn_sched_barrier(0);
      quad_store<GRP, GLU, HALF ? 32 : 16, PAST>(acc, gr, bias, Y, ldy, cur.m0 + (HALF ? 16 : 128) * wr, cur.n0 + wc * 128, cur.M, N, li, g, sw, !full);
      if (ahead < 0) break;
      ahead = after;
      cur = next, next = then;
      if constexpr (GATHER) {
#pragma unroll
        for (int i = 0; i < 8; ++i) vx[i] = vn[i], vn[i] = offset_of(pairs[i], i);
      }
#pragma unroll
      for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("s_nop 7" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#undef Q_MFMA
#undef Q_FOUR
#undef Q_UPPER8
#undef Q_X
#undef Q_W
#undef Q_LOAD
#undef Q_RSRC
  __builtin_amdgcn_s_waitcnt(0x0070);  // no load of this wave is on its way into LDS any more,
  if constexpr (RING) return;
  const int m0 = cur.m0, n0 = cur.n0;
  M = cur.M;
  __builtin_amdgcn_s_barrier();  // and all waves are there
  __builtin_amdgcn_sched_barrier(0);
  // Out through LDS, 64 columns of the wave's 128 rows at a time as fp32. A lane holds, of row 16 mt + li, eight neighbouring columns in tiles
  // 2 p and 2 p + 1. The bf16 stores bypass the caches' replacement, which keeps X and W of the tiles to come: 632 -> 606 us at 8192 x 12288 x
  // 4096, 1.5 % of a prompt step.
  char* img = smem + w * BUF;
  if constexpr (QKV) {
    const int D = qe.D, nq = qe.nh * D, nqk = nq + qe.nkv * D, rh = qe.rot >> 1, nw0 = n0 + wc * 128, mw0 = m0 + wr * 128;
    const bool rope = qe.do_rope != 0 && nw0 < nqk, cached = qe.kc != nullptr && nw0 + 127 >= nq;
    int* rpos = reinterpret_cast<int*>(smem + 4 * BUF + w * 2048);                  // [128] the rows' positions
    int64_t* rbase = reinterpret_cast<int64_t*>(smem + 4 * BUF + w * 2048 + 512);  // [128] and first numbers in the cache, -1: not cached
    int64_t ps[2] = {0, 0}, sl[2] = {-1, -1};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = min(mw0 + lane + 64 * i, M - 1);
      if (rope) ps[i] = qe.pos[m];
      if (cached) sl[i] = qe.slot[m];
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int n = nw0 + 32 * p + 8 * g;
      float b[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (bias && n < N) {
#pragma unroll
        for (int i = 0; i < 8; ++i) b[i] = bf2f(bias[n + i]);
      }
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) {
        u16x8 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          o[i] = f2bf(acc[2 * p][mt][i] + b[i]);
          o[4 + i] = f2bf(acc[2 * p + 1][mt][i] + b[4 + i]);
        }
        *reinterpret_cast<u16x8*>(img + (16 * mt + li) * 256 + (((4 * p + g) ^ li) << 4)) = o;
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      rpos[lane + 64 * i] = (int)ps[i];
      const unsigned u = (unsigned)sl[i], bs = (unsigned)qe.block_size, blk = u / bs;
      rbase[lane + 64 * i] = sl[i] < 0 ? -1 : ((int64_t)blk * qe.nkv * bs + (u - blk * bs)) * D;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int c = lane & 15, n = nw0 + 8 * c, d = n % D;
    const bool is_v = n >= nqk, turn = rope && !is_v && d < qe.rot, keep = cached && n >= nq && n < N;
    bf16_t* const cache = (is_v ? qe.vc : qe.kc) + (int64_t)((n - (is_v ? nqk : nq)) / D) * qe.block_size * D + d;
    const int a = turn ? d >> 1 : 0;  // (columns that do not turn read an angle that nobody uses)
    constexpr int U = 4;
#pragma unroll 1
    for (int i0 = 0; i0 < 32; i0 += U) {
      f32x4 cs[U], sn[U];
      if (rope) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t at = (int64_t)rpos[4 * (i0 + u) + g] * rh + a;
          cs[u] = *reinterpret_cast<const f32x4*>(qe.cos_t + at);
          sn[u] = *reinterpret_cast<const f32x4*>(qe.sin_t + at);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = 4 * (i0 + u) + g, m = mw0 + r;
        u16x8 o = *reinterpret_cast<const u16x8*>(img + r * 256 + ((c ^ (r & 15)) << 4));
        if (turn) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = bf2f(o[2 * i]), y = bf2f(o[2 * i + 1]);
            o[2 * i] = f2bf(x * cs[u][i] - y * sn[u][i]);
            o[2 * i + 1] = f2bf(y * cs[u][i] + x * sn[u][i]);
          }
        }
        if (m >= M || n >= N) continue;
        __builtin_nontemporal_store(o, reinterpret_cast<u16x8*>(Y + (int64_t)m * ldy + n));
        const int64_t base = rbase[r];
        if (keep && base >= 0) __builtin_nontemporal_store(o, reinterpret_cast<u16x8*>(cache + base));
      }
    }
    return;
  }
  auto flush = [&](int c0) {  // the image is columns c0 .. c0 + 63 of the output
    const int j = lane & 7, n = c0 + 8 * j;
    float bl[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (bias && n < N) {
#pragma unroll
      for (int i = 0; i < 8; ++i) bl[i] = bf2f(bias[n + i]);
    }
    auto some = [&](auto kind) {
#pragma unroll 2
      for (int i = 0; i < 16; ++i) {
        const int r = 8 * i + (lane >> 3), m = m0 + wr * 128 + r;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(img + r * 256 + (((2 * j) ^ (r & 15)) << 4));
        const f32x4 hi = *reinterpret_cast<const f32x4*>(img + r * 256 + (((2 * j + 1) ^ (r & 15)) << 4));
        u16x8 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = f2bf(apply_act(lo[e] + bl[e], kind()));
          o[4 + e] = f2bf(apply_act(hi[e] + bl[4 + e], kind()));
        }
        if (m < M && n < N) __builtin_nontemporal_store(o, reinterpret_cast<u16x8*>(Y + (int64_t)m * ldy + n));
      }
    };
    // (a loop for each function: with the choice inside, the unrolled code does not fit the instruction cache)
    if (act == ACT_GELU_TANH) some(std::integral_constant<int, ACT_GELU_TANH>());
    else if (act == ACT_GELU) some(std::integral_constant<int, ACT_GELU>());
    else if (act == ACT_RELU) some(std::integral_constant<int, ACT_RELU>());
    else some(std::integral_constant<int, ACT_RELU2>());
  };
  auto put = [&](int p, const f32x4 (&lo)[8], const f32x4 (&hi)[8]) {
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      char* row = img + (16 * mt + li) * 256;
      const int c = 8 * (p & 1) + 2 * g;
      *reinterpret_cast<f32x4*>(row + ((c ^ li) << 4)) = lo[mt];
      *reinterpret_cast<f32x4*>(row + (((c + 1) ^ li) << 4)) = hi[mt];
    }
  };
  // the image passes numbers between the lanes of this wave: its writes before the reads, and those before the next writes
  auto turn = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  put(0, acc[0], acc[1]);
  put(1, acc[2], acc[3]);
  turn();
  flush(n0 + wc * 128);
  turn();
  put(2, acc[4], acc[5]);
  put(3, acc[6], acc[7]);
  turn();
  flush(n0 + wc * 128 + 64);
}

// rows: of X that one descriptor covers; es: bytes of an output element; list: tiles of an expert list, whose waves' rows alternate (quad_store)
bool gemm_quad_ok(int N, int K, int64_t ldx, int64_t ldw, int64_t rows, const void* Y, int64_t ldy, int es, bool glu, bool list) {
  return K % 64 == 0 && K >= 64 && (uint64_t)rows * (uint64_t)ldx * 2 < (1ull << 31) && (uint64_t)256 * (uint64_t)ldw * 2 < (1ull << 31) &&
         ldx % 8 == 0 && ldw % 8 == 0 && N % (glu ? 32 : 8) == 0 && ((uintptr_t)Y & 15) == 0 && ldy * es % 16 == 0 &&
         (uint64_t)(list ? 240 : 128) * (uint64_t)ldy * es < (1ull << 31);
}

void launch_gemm_quad(int grp, const bf16_t* X, int64_t ldx, const bf16_t* W, int64_t ldw, const bf16_t* bias, bf16_t* Y,
                      int64_t ldy, int M, int N, int K, int act, int glu, int group_m, unsigned nwg, const PpGroup& gr,
                      hipStream_t st, const QkvEpi* qe) {
  // a workgroup per CU, each taking every 256th tile; rings of fewer than four steps do not reach into another tile
  const unsigned ring = K >= 256 ? std::min(nwg, 256u) : nwg;
  const bool lds = qe || (!glu && grp != 2 && act != ACT_NONE);
  // fp32 sums of up to 128 MB stay in the caches. us, three launches, past them and in them: 5554 pairs x 2048 (45 MB), 8 experts of 1024, 124 and 118;
  // 11108 x 2048 (91 MB), 16 of 768, 204 and 195; 22216 x 1024, 128 of 256, 128 and 117; 32768 x 1024 (134 MB), 32 of 512, 205 and 196; 16384 x 2048,
  // 8 of 1024, 302 and 305; 22216 x 2048 (182 MB), 64 of 768, 400 and 420; 65536 x 1024, 128 of 256, 284 and 295. (A list of P pairs has room for
  // ceil(P / 256) + E tiles.)
  const bool past = (int64_t)std::max(gr.maxt - gr.E, 1) * 256 * ldy * 4 > (128 << 20);
#define LAUNCH_P(G_, U_, Q_, R_, P_) \
  gemm_quad_kernel<G_, U_, Q_, R_, P_><<<R_ ? ring : nwg, 256, 0, st>>>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, act, group_m, gr, qe ? *qe : QkvEpi{})
#define LAUNCH_Q(G_, U_, Q_, R_) LAUNCH_P(G_, U_, Q_, R_, true)
  if (qe) LAUNCH_Q(0, 0, true, false);
  else if (grp == 2 && past) LAUNCH_Q(2, 0, false, true);
  else if (grp == 2) LAUNCH_P(2, 0, false, true, false);
  else if (grp == 3) LAUNCH_Q(3, 1, false, true);
  else if (grp == 1 && glu) LAUNCH_Q(1, 1, false, true);
  else if (grp == 1 && lds) LAUNCH_Q(1, 0, false, false);
  else if (grp == 1) LAUNCH_Q(1, 0, false, true);
  else if (glu && act == ACT_GELU_TANH) LAUNCH_Q(0, 2, false, true);
  else if (glu) LAUNCH_Q(0, 1, false, true);
  else if (lds) LAUNCH_Q(0, 0, false, false);
  else LAUNCH_Q(0, 0, false, true);
#undef LAUNCH_Q
#undef LAUNCH_P
  HIP_CHECK_LAUNCH();
}
