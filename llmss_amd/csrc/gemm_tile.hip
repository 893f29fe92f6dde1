// bf16 matrix products on the matrix cores for the shapes gemm.hip's plans do not cover: batched per-head products
// over strided views, products that keep an fp32 output, and the grouped expert GEMMs of a mixture-of-experts layer
// (row gather, per-expert weights, the clamped gated activation fused behind the gate / up product).
//
//   C[b][m][n] = sum_k A[b][m][k] * B[b][n][k] (+ bias[n])        A, B bf16 with k contiguous; C bf16 or fp32
//
// One 64x64 or 128x128 output tile per 256-thread workgroup, k in steps of 64 through LDS, v_mfma_f32_16x16x32_bf16.
// Fragment layout: lane (li = lane % 16, g = lane / 16) holds k = 8g .. 8g + 7 of row li
// (A) or of column li (B); the accumulator holds rows 4g .. 4g + 3 of column li. Rows, columns and the k tail are
// bounds-checked while staging (zero fill), so any M, N, K works; rows that are 16-byte aligned take vector loads.
//
// Modes: PLAIN (batched, strided), GATE_UP (grouped: rows of an expert's tile list, A rows gathered through
// order[] / top, two weight matrices, output glu(gate, up) in bf16), UP (the same with one weight matrix, output
// gelu(up), the error-function form) and DOWN (grouped: A = the activation rows,
// fp32 output). The tile list and offsets are those moe_group writes (moe.hip).
#include <cmath>

#include "anytype.h"
#include "gemm_quad.h"

#define GT_BK 64
#define GT_LD 72  // bf16 per LDS row: 144 bytes, keeps ds_read_b128 rows 16-byte aligned and spreads the banks

enum { GT_PLAIN = 0, GT_GATE_UP = 1, GT_DOWN = 2, GT_UP = 3 };

struct GemmTileArgs {
  const bf16_t* A;
  const bf16_t* B;
  const bf16_t* B2;  // GATE_UP: the up weights
  void* C;
  int M, N, K;
  int64_t sAb, sAm, sBb, sBn, sCb, sCm;
  // grouped modes
  const int* meta;
  const int* order;
  int E, maxt, top;
  float limit, alpha;
  const float* pw;  // GATE_UP: weight of each (token, slot) pair on the expert's input (null: 1)
  int silu;         // GATE_UP: silu(g) * u instead of the clamped form
  int ilv;          // GATE_UP: one weight matrix, gate and up rows in alternating groups of 16 (B the first gate row, B2 the first up row)
  const bf16_t* bias;  // PLAIN: [N] or null
  int wide;            // PLAIN, bf16 results in the ring kernel: rows and columns in pieces of 16 bytes
};

// 8 consecutive k of one row (zero beyond the row / k range)
__device__ __forceinline__ u16x8 gt_load(const bf16_t* row, int k, int K, bool vec) {
  u16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (row) {
    if (vec && k + 8 <= K) {
      v = *reinterpret_cast<const u16x8*>(row + k);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (k + i < K) v[i] = row[k + i];
    }
  }
  return v;
}

// BM x BN output tile per 256-thread workgroup (64x64, 128x128, or 128x256 where LDS reads would otherwise bound it), waves in a 2x2 grid: each wave owns a
// (BM/2) x (BN/2) block = MB x NB accumulators of 16x16. Per 32 of k a wave reads MB A fragments and NB B
// fragments from LDS for MB * NB MFMAs (two such halves per staged k step of 64). The next k step's global loads are issued into registers before the current
// step's MFMAs and written to LDS after them, so memory latency overlaps the matrix work.
template <int MODE, typename TC, int BM, int BN>
__global__ __launch_bounds__(256, BM * BN > 128 * 128 ? 2 : 1) void gemm_tile_kernel(GemmTileArgs p) {
  constexpr int MB = BM / 32, NB = BN / 32;   // 16x16 blocks per wave, rows x columns
  constexpr int CA = BM / 32, CB = BN / 32;   // 16-byte chunks per thread per staged tile
  constexpr bool DUAL = MODE == GT_GATE_UP;
  __shared__ __attribute__((aligned(16))) bf16_t As[BM * GT_LD];
  __shared__ __attribute__((aligned(16))) bf16_t Bs[BN * GT_LD];
  __shared__ __attribute__((aligned(16))) bf16_t B2s[DUAL ? BN * GT_LD : 8];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, g = lane >> 4;
  const int wm = (w >> 1) * (BM / 2), wn = (w & 1) * (BN / 2);
  int n0 = blockIdx.x * BN;
  int m0 = 0, rows = 0, crow0 = 0;
  const bf16_t* A = p.A;
  const bf16_t* B = p.B;
  const bf16_t* B2 = p.B2;
  if constexpr (MODE == GT_PLAIN) {
    m0 = blockIdx.y * BM;
    rows = min(BM, p.M - m0);
    A += (int64_t)blockIdx.z * p.sAb;
    B += (int64_t)blockIdx.z * p.sBb;
  } else {
    if ((int)blockIdx.y >= p.meta[0]) return;
    // every die takes a contiguous run of the list's tiles, all their column tiles with them: an expert's weights then
    // pass through few L2s, and a row tile's rows stay in one
    const int id = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, p.meta[0] * gridDim.x);
    const int ty = id / gridDim.x;
    n0 = (id % gridDim.x) * BN;
    const int e = p.meta[1 + (p.E + 1) + ty];
    crow0 = p.meta[1 + (p.E + 1) + p.maxt + ty];
    rows = min(BM, p.meta[1 + e + 1] - crow0);
    B += (int64_t)e * p.sBb;
    if constexpr (DUAL) B2 += (int64_t)e * p.sBb;
  }
  // staging: chunk c = tid + 256 i -> (row c / 8, k offset (c % 8) * 8) of each tile
  const bf16_t* arow[CA];
  const bf16_t* brow[CB];
  const bf16_t* b2row[CB];
  bool avec[CA], bvec[CB], b2vec[CB];
  const int sk = (tid & 7) * 8;
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int sr = (tid >> 3) + 32 * i;
    arow[i] = nullptr;
    if (sr < rows) {
      if constexpr (MODE == GT_PLAIN) arow[i] = A + (int64_t)(m0 + sr) * p.sAm;
      else if constexpr (MODE == GT_GATE_UP || MODE == GT_UP) arow[i] = A + (int64_t)(p.order[crow0 + sr] / p.top) * p.sAm;
      else arow[i] = A + (int64_t)(crow0 + sr) * p.sAm;
    }
    avec[i] = arow[i] && ((uintptr_t)arow[i] & 15) == 0;
  }
#pragma unroll
  for (int i = 0; i < CB; ++i) {
    const int sr = (tid >> 3) + 32 * i;
    int nr = n0 + sr;  // row of the weights
    if constexpr (DUAL) nr = p.ilv ? (nr >> 4) * 32 + (nr & 15) : nr;
    brow[i] = (n0 + sr < p.N) ? B + (int64_t)nr * p.sBn : nullptr;
    bvec[i] = brow[i] && ((uintptr_t)brow[i] & 15) == 0;
    b2row[i] = nullptr;
    b2vec[i] = false;
    if constexpr (DUAL) {
      b2row[i] = (n0 + sr < p.N) ? B2 + (int64_t)nr * p.sBn : nullptr;
      b2vec[i] = b2row[i] && ((uintptr_t)b2row[i] & 15) == 0;
    }
  }
  u16x8 ra[CA], rb[CB], rb2[CB];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CA; ++i) ra[i] = gt_load(arow[i], k0 + sk, p.K, avec[i]);
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      rb[i] = gt_load(brow[i], k0 + sk, p.K, bvec[i]);
      if constexpr (DUAL) rb2[i] = gt_load(b2row[i], k0 + sk, p.K, b2vec[i]);
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < CA; ++i) *reinterpret_cast<u16x8*>(&As[((tid >> 3) + 32 * i) * GT_LD + sk]) = ra[i];
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      *reinterpret_cast<u16x8*>(&Bs[((tid >> 3) + 32 * i) * GT_LD + sk]) = rb[i];
      if constexpr (DUAL) *reinterpret_cast<u16x8*>(&B2s[((tid >> 3) + 32 * i) * GT_LD + sk]) = rb2[i];
    }
  };

  f32x4 acc[MB][NB], acc2[DUAL ? MB : 1][DUAL ? NB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (DUAL) acc2[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  fetch(0);
  for (int k0 = 0; k0 < p.K; k0 += GT_BK) {
    __syncthreads();  // the previous step's fragment reads are done
    stash();
    __syncthreads();
    if (k0 + GT_BK < p.K) fetch(k0 + GT_BK);
#pragma unroll
    for (int ks = 0; ks < GT_BK; ks += 32) {
      s16x8 a[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i)
        a[i] = *reinterpret_cast<const s16x8*>(&As[(wm + 16 * i + li) * GT_LD + ks + 8 * g]);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const s16x8 b = *reinterpret_cast<const s16x8*>(&Bs[(wn + 16 * j + li) * GT_LD + ks + 8 * g]);
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b, acc[i][j], 0, 0, 0);
        if constexpr (DUAL) {
          const s16x8 b2 = *reinterpret_cast<const s16x8*>(&B2s[(wn + 16 * j + li) * GT_LD + ks + 8 * g]);
#pragma unroll
          for (int i = 0; i < MB; ++i)
            acc2[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b2, acc2[i][j], 0, 0, 0);
        }
      }
    }
  }
  TC* C = (TC*)p.C;
  if constexpr (MODE == GT_PLAIN) C += (int64_t)blockIdx.z * p.sCb;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = wm + 16 * i + 4 * g + q;
      if (r >= rows) continue;
      TC* crow = C + (int64_t)((MODE == GT_PLAIN ? m0 : crow0) + r) * p.sCm;
      float sw = 1.0f;
      if constexpr (MODE == GT_GATE_UP || MODE == GT_UP) sw = p.pw ? p.pw[p.order[crow0 + r]] : 1.0f;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int n = n0 + wn + 16 * j + li;
        if (n >= p.N) continue;
        float v = acc[i][j][q];
        if constexpr (DUAL) v = glu_clamped_t(v * sw, acc2[i][j][q] * sw, p.limit, p.alpha, p.silu);
        if constexpr (MODE == GT_UP) v = gelu_erf(v * sw);
        if constexpr (MODE == GT_PLAIN) v += p.bias ? bf2f(p.bias[n]) : 0.f;
        El<TC>::st(crow + n, v);
      }
    }
}

// Products with whole k-steps and rows of 16-byte alignment: as above, but operands go straight to a ring of NS k-steps in
// LDS, NS - 1 of them on their way, one barrier a step; 8 rows x 128 bytes a load, chunks XOR-swizzled by row so that fragment reads meet
// no bank conflict. Bound by the weights of the experts that the tokens reach and, with few rows each, by the latency of a step: the kernel
// above waits out one step's loads after each, its two barriers between them. Experts start at different k-steps (e * 11): rows of a power of
// two bytes lie on few memory channels, which all tiles would otherwise walk together (32 experts of 768 x 2048, 80 rows each: 100 -> 94 us of
// both products; by row tile instead, tiles that share an expert's weights lose each other: 188 rows each 151 -> 158). us of both products
// against the kernel above: 16 experts of 512 x 1024, 38 rows each 33.2 -> 24.6; 32 of 768 x 2048, 80 rows 120 -> 94, 103 rows 117 -> 99; 64 of
// 1408 x 2048, 96 rows 360 -> 294, 66 rows 321 -> 277; but 89 against 82 for 64 of 896 x 768, 55 rows each: moe_plan below says
// which layers come here. Batched and 32-bit-result products (PLAIN), whose K of 128 - 256 is on its way whole and whose bf16 results leave in 16-byte pieces
// instead of two bytes a lane: 16 heads of 8261 x 256 x 128 45.5 -> 35.6 us, x 128 x 256 37.8 -> 28.4, one of 8261 x 4096 x 1024 in 32 bits 143 -> 112,
// 64 x 2048 x 2048 23.2 -> 11.6, 8 x 2048 x 1024 12.2 -> 7.3. Four or six steps were slower everywhere (822 x 4 rows over 32 experts: 127 and 139
// against 120). 128 rows: 128 x 128 tiles for one matrix (64 and 256 columns 111 and 105 against 102 us).
template <int MODE, typename TC, int BM, int BN, int NS>
__global__ __launch_bounds__(256) void tile_ring_kernel(GemmTileArgs p) {
  constexpr int MB = BM / 32, NB = BN / 32;
  constexpr bool DUAL = MODE == GT_GATE_UP;
  constexpr int AI = BM / 32, BI = (DUAL ? 2 : 1) * BN / 32;  // 1-KiB loads (8 rows of a k-step) of a wave
  constexpr int LOADS = AI + BI, SLOT = (BM + (DUAL ? 2 : 1) * BN) * 128;
  static_assert(NS * SLOT <= 160 * 1024 && (NS - 2) * LOADS <= 63, "LDS and the wait's immediate");
  __shared__ __attribute__((aligned(16))) char smem[NS * SLOT];
  const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (w >> 1) * (BM / 2), wn = (w & 1) * (BN / 2);
  constexpr bool PLAIN = MODE == GT_PLAIN;
  int n0 = blockIdx.x * BN, e = blockIdx.z, crow0 = blockIdx.y * BM, rows = min(BM, p.M - crow0);
  const bf16_t* A = p.A;
  if constexpr (PLAIN) {
    A += (int64_t)e * p.sAb + (int64_t)crow0 * p.sAm;
  } else {
    if ((int)blockIdx.y >= p.meta[0]) return;
    const int id = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, p.meta[0] * gridDim.x);
    const int ty = id / gridDim.x;
    n0 = (id % gridDim.x) * BN;
    e = p.meta[1 + (p.E + 1) + ty], crow0 = p.meta[1 + (p.E + 1) + p.maxt + ty];
    rows = min(BM, p.meta[1 + e + 1] - crow0);
  }

  const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(A)), (short)0, 0x7fffffff, 0x00020000);
  // PLAIN: of B too from the tile's own first row on, so that 31 bits hold a tile's rows whatever the matrix's size
  const int b0 = PLAIN ? n0 : 0;
  const auto rb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(p.B + (int64_t)e * p.sBb + (int64_t)b0 * p.sBn)), (short)0, 0x7fffffff, 0x00020000);
  const auto rb2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>((DUAL ? p.B2 : p.B) + (int64_t)e * p.sBb)),
                                                     (short)0, 0x7fffffff, 0x00020000);
  // wave w takes rows 8 (w + 4 i) .. + 7 of each operand; past the rows or columns, or past the last step: an offset that reads as zero (past
  // both the two offsets wrap to the operand's first bytes, which are there and land where nobody reads)
  uint32_t va[AI], vb[BN / 32];
  const int sr0 = 8 * w + (lane >> 3), ch = ((lane & 7) ^ (sr0 & 7)) << 4;
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int sr = sr0 + 32 * i;
    va[i] = 0x80000000u;
    if (sr < rows) {
      const int row = PLAIN ? sr : MODE == GT_DOWN ? crow0 + sr : p.order[crow0 + sr] / p.top;
      va[i] = (uint32_t)(row * p.sAm * 2 + ch);
    }
  }
#pragma unroll
  for (int i = 0; i < BN / 32; ++i) {
    const int n = n0 + sr0 + 32 * i, row = DUAL && p.ilv ? (n >> 4) * 32 + (n & 15) : n - b0;
    vb[i] = n < p.N ? (uint32_t)(row * p.sBn * 2 + ch) : 0x80000000u;
  }
  const int nk = p.K / 64;
  const int k0 = PLAIN ? 0 : (e * 11) % nk;
#define MR_ISSUE(T_, S_)                                                                                                          \
  do {                                                                                                                            \
    const int q_ = (T_) + k0 >= nk ? (T_) + k0 - nk : (T_) + k0;                                                                   \
    const uint32_t so_ = (T_) < nk ? (uint32_t)q_ * 128u : 0x80000000u;                                                         \
    char* sl_ = smem + (S_) * SLOT + w * 1024;                                                                                    \
    _Pragma("unroll") for (int i_ = 0; i_ < AI; ++i_)                                                                             \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_AS void*)(sl_ + i_ * 4096), 16, (uint32_t)(va[i_] + so_), 0, 0, 0);       \
    _Pragma("unroll") for (int i_ = 0; i_ < BN / 32; ++i_)                                                                        \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LDS_AS void*)(sl_ + BM * 128 + i_ * 4096), 16, (uint32_t)(vb[i_] + so_), 0, 0, 0); \
    if (DUAL) _Pragma("unroll") for (int i_ = 0; i_ < BN / 32; ++i_)                                                              \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb2, (LDS_AS void*)(sl_ + (BM + BN) * 128 + i_ * 4096), 16, (uint32_t)(vb[i_] + so_), 0, 0, 0); \
  } while (0)
  f32x4 acc[MB][NB], acc2[DUAL ? MB : 1][DUAL ? NB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (DUAL) acc2[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) MR_ISSUE(s, s);
  const int x0 = (g ^ (li & 7)) << 4, x1 = ((4 + g) ^ (li & 7)) << 4;
  int slot = 0;
  for (int t = 0; t < nk; ++t) {
    // this wave's part of step t is there, and its reads of step t - 1 are done
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * LOADS) : "memory");
    __builtin_amdgcn_s_barrier();  // every wave's
    asm volatile("" ::: "memory");
    MR_ISSUE(t + NS - 1, slot == 0 ? NS - 1 : slot - 1);  // into the slot of step t - 1
    const char* st = smem + slot * SLOT;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int xo = s ? x1 : x0;
      s16x8 a[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) a[i] = *reinterpret_cast<const s16x8*>(st + (wm + 16 * i + li) * 128 + xo);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const s16x8 b = *reinterpret_cast<const s16x8*>(st + (BM + wn + 16 * j + li) * 128 + xo);
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b, acc[i][j], 0, 0, 0);
        if constexpr (DUAL) {
          const s16x8 b2 = *reinterpret_cast<const s16x8*>(st + (BM + BN + wn + 16 * j + li) * 128 + xo);
#pragma unroll
          for (int i = 0; i < MB; ++i) acc2[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b2, acc2[i][j], 0, 0, 0);
        }
      }
    }
    slot = slot == NS - 1 ? 0 : slot + 1;
  }
#undef MR_ISSUE
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (loads past the last step write to LDS too)
  TC* C = (TC*)p.C;
  if constexpr (PLAIN) C += (int64_t)e * p.sCb;
  if constexpr (PLAIN && sizeof(TC) == 2) {
    if (p.wide) {  // bf16 results in whole 16-byte pieces, through LDS
      constexpr int LD = BN + 8;
      static_assert(BM * LD * 2 <= NS * SLOT, "the tile's image");
      bf16_t* im = reinterpret_cast<bf16_t*>(smem);
      __syncthreads();  // every wave's fragment reads are done
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int n = n0 + wn + 16 * j + li;
          const float b = p.bias && n < p.N ? bf2f(p.bias[n]) : 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) El<TC>::st(im + (wm + 16 * i + 4 * g + q) * LD + wn + 16 * j + li, acc[i][j][q] + b);
        }
      __syncthreads();
      for (int c = threadIdx.x; c < BM * BN / 8; c += 256) {
        const int row = c / (BN / 8), col = c % (BN / 8) * 8;
        if (row < rows && n0 + col < p.N)
          *reinterpret_cast<u16x8*>(C + (int64_t)(crow0 + row) * p.sCm + n0 + col) = *reinterpret_cast<const u16x8*>(im + row * LD + col);
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = wm + 16 * i + 4 * g + q;
      if (r >= rows) continue;
      TC* crow = C + (int64_t)(crow0 + r) * p.sCm;
      float sw = 1.0f;
      if constexpr (MODE != GT_DOWN && !PLAIN) sw = p.pw ? p.pw[p.order[crow0 + r]] : 1.0f;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int n = n0 + wn + 16 * j + li;
        if (n >= p.N) continue;
        float v = acc[i][j][q];
        if constexpr (DUAL) v = glu_clamped_t(v * sw, acc2[i][j][q] * sw, p.limit, p.alpha, p.silu);
        if constexpr (MODE == GT_UP) v = gelu_erf(v * sw);
        if constexpr (PLAIN) v += p.bias ? bf2f(p.bias[n]) : 0.f;
        El<TC>::st(crow + n, v);
      }
    }
}

static int plain_tile(int M, int N) { return M >= 512 && N >= 128 ? 128 : 64; }  // big tiles where there is enough work to fill the chip

// Whether a batched or 32-bit-result product of whole k-steps takes the ring: not on 64 x 64 tiles that do not all run at once, three on a CU there,
// where the kernel without it has more of them - up to half a wave too many, and with K up to 256 any number. Over 1900 products of 769 tiles and more
// the ring took 1.04 - 1.25 of that kernel's time at K = 64 - 192, 1.01 - 1.05 up to 1152 tiles beyond, else 0.95 (tiles of 128 x 128: 0.83, 0.94 in 32
// bits, hardly one slower). us without and with: 16 heads of 3680 x 40 x 128 in 32 bits 8.3 and 9.9, 8 of 383 x 2040 x 192 14.5 and 17.6, 40 of 8 x
// 3936 x 64 10.3 and 14.3. With this line 0.80 over 4477 other products, 94 above 1.02, 1.12 at worst (64 of 7594 x 103 x 320 173 and 194).
bool gemm_tile_rings(int M, int N, int K, int batch) {
  const int T = plain_tile(M, N);
  const int64_t tiles = (int64_t)((M + T - 1) / T) * ((N + T - 1) / T) * batch;
  return K % 64 == 0 && (T == 128 || tiles <= 768 || (K > 256 && tiles > 1152));
}

void launch_gemm_tile(const void* A, const void* B, void* C, int M, int N, int K, int batch, int64_t sAb, int64_t sAm,
                      int64_t sBb, int64_t sBn, int64_t sCb, int64_t sCm, int dc, const void* bias, hipStream_t st) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  const int T = plain_tile(M, N);
  if (batch > 65535 || (M + T - 1) / T > 65535) throw std::runtime_error("gemm_tile: grid too large");
  GemmTileArgs a{};
  a.A = (const bf16_t*)A; a.B = (const bf16_t*)B; a.C = C;
  a.M = M; a.N = N; a.K = K;
  a.sAb = sAb; a.sAm = sAm; a.sBb = sBb; a.sBn = sBn; a.sCb = sCb; a.sCm = sCm;
  a.bias = (const bf16_t*)bias;
  dim3 g((N + T - 1) / T, (M + T - 1) / T, batch);
  if (dc != 0 && dc != 1) throw std::runtime_error("gemm_tile: bad output dtype code");
  // whole k-steps, rows of 16-byte alignment of which a tile's 128, of either operand, fit 31 bits: the ring, where the size is one for it
  const bool ring = gemm_tile_rings(M, N, K, batch) && K > 0 && !((sAb | sAm | sBb | sBn) & 7) && !(((uintptr_t)A | (uintptr_t)B) & 15) && sAm >= 0 && sBn >= 0 &&
                    std::max(sAm, sBn) < (1 << 22) && K < (1 << 22);
  if (ring) {
    a.wide = N % 8 == 0 && !((sCb | sCm) & 7) && !((uintptr_t)C & 15);
    if (T == 128) {
      if (dc == 0) tile_ring_kernel<GT_PLAIN, bf16_t, 128, 128, 2><<<g, 256, 0, st>>>(a);
      else tile_ring_kernel<GT_PLAIN, float, 128, 128, 2><<<g, 256, 0, st>>>(a);
    } else {
      if (dc == 0) tile_ring_kernel<GT_PLAIN, bf16_t, 64, 64, 3><<<g, 256, 0, st>>>(a);
      else tile_ring_kernel<GT_PLAIN, float, 64, 64, 3><<<g, 256, 0, st>>>(a);
    }
    HIP_CHECK_LAUNCH();
    return;
  }
  if (T == 128) {
    if (dc == 0) gemm_tile_kernel<GT_PLAIN, bf16_t, 128, 128><<<g, 256, 0, st>>>(a);
    else gemm_tile_kernel<GT_PLAIN, float, 128, 128><<<g, 256, 0, st>>>(a);
  } else {
    if (dc == 0) gemm_tile_kernel<GT_PLAIN, bf16_t, 64, 64><<<g, 256, 0, st>>>(a);
    else gemm_tile_kernel<GT_PLAIN, float, 64, 64><<<g, 256, 0, st>>>(a);
  }
  HIP_CHECK_LAUNCH();
}

// The ring kernel takes whole k-steps, 16-byte rows, and operands whose places fit 31 bits (`rows`: an upper bound of A's)
static bool moe_ring_ok(const GemmTileArgs& a, int64_t lda, int64_t rows, int64_t wrows) {
  return a.K % 64 == 0 && a.K > 0 && lda % 8 == 0 && !(((uintptr_t)a.A | (uintptr_t)a.B | (uintptr_t)a.B2) & 15) &&
         (rows + 1) * lda * 2 < (1ll << 31) && wrows * a.K * 2 < (1ll << 31);
}

// 64-row tiles: three steps deep where the list's tiles (a row tile an expert, or half of one beside the full ones) then still run at once,
// else two.
template <int MODE, typename TC>
static void moe_ring64(const GemmTileArgs& a, hipStream_t st) {
  constexpr int slot = MODE == GT_GATE_UP ? 24 : 16;  // KB
  constexpr int at3 = 256 * (160 / (3 * slot));
  const int cols = (a.N + 63) / 64;
  const int64_t tiles = (int64_t)std::max(std::min(a.E, a.maxt), a.maxt - a.E / 2) * cols;
  const dim3 g(cols, a.maxt);
  if (tiles <= at3) tile_ring_kernel<MODE, TC, 64, 64, 3><<<g, 256, 0, st>>>(a);
  else tile_ring_kernel<MODE, TC, 64, 64, 2><<<g, 256, 0, st>>>(a);
}

// Rows of a tile for a layer of experts (more than 8 pairs each) whose operands the ring kernel takes, and whether its products take that kernel
// (bit 0: gate and up, bit 1: down; 128 rows: always). `rows`: what the rule without the ring says, 64 below 128 pairs an expert, 128 from there on,
// 256 (gemm_quad.hip) where `big` and from 128 pairs on (gate and up in two matrices: 256). That stays unless another form is priced 1.12 times below,
// and the kernel without the ring, for a product of 64 rows, unless the ring is priced 1.08 times below.
// A product's price: `at_once` of its tiles share a CU, a step of 64 of k then taking `step` us and `more` for every tile beside the first, behind
// `begin` a tile; and its weights at `rate`, the two joined as sides of a right triangle (neither hides the other). Beside the products a start, the
// rows that are gathered, written and read, and the pairs' grouping. Experts get as many rows as if tokens chose at random. Constants fitted over two thirds
// of 1020 random layers (2 - 200 experts of 64 - 3072 x 128 - 3072, 9 - 600 pairs each, gate and up together, apart or no gate, weights from
// memory), 4 - 8 % off on average on the other third.
// Against that rule, over 900 other layers, a third of them with uneven experts: 0.737 of the whole layer's time, five above 1.02, 1.09 at worst (198
// experts of 192 x 384, uneven, 71 pairs each 50 -> 54 us). By tile counts alone instead of prices, 128 rows from 64 pairs an expert and 384 tiles on: 0.79 over
// 1020, 54 above 1.02, 1.35 at worst (142 of 768 x 128, 70 pairs each 57 -> 77; now 64 rows, 53 there and here). us without and with: 64 of 896 x 768,
// 55 pairs each 82 and 89 (stays); 12 of 2176 x 512, 123 each 65 -> 47; 64 of 1408 x 2048, 96 each 405 -> 373.
struct MoeCost {  // us; bytes per us
  int rows;
  double start, rate, row_rate, pair;
  struct {
    double step, more, begin;
    int at_once, bn;
  } plain, glu;
};
static constexpr MoeCost kMoeCost[] = {
    {64, 14.0, 5.25e6, 5.72e6, 0.243e-3, {0.894, 0.070, 0.0, 5, 64}, {0.999, 0.178, 0.90, 4, 64}},     // without the ring
    {64, 14.2, 4.93e6, 5.11e6, 0.298e-3, {0.367, 0.213, 0.0, 5, 64}, {0.411, 0.372, 1.33, 3, 64}},     // with it
    {128, 16.3, 5.87e6, 4.59e6, 0.545e-3, {0.936, 0.127, 2.03, 2, 128}, {0.720, 0.483, 0.55, 2, 64}},
    {256, 9.67, 5.16e6, 12.7e6, 0.646e-3, {1.350, 0.0, 13.5, 1, 256}, {1.190, 0.0, 6.94, 1, 128}}};
void moe_plan(int P, int E, int F, int N, int K, bool glu, int rows, bool big, int* rows_out, int* ring) {
  auto row_tiles = [&](int r) {
    const double mean = (double)P / E;
    double t = 0;
    for (double q : {-1.5, -0.9, -0.5, -0.15, 0.15, 0.5, 0.9, 1.5}) t += std::ceil(std::max(1.0, mean + q * std::sqrt(mean)) / r);
    return t * E / 8;
  };
  auto us = [&](const MoeCost& c, bool up) {
    const auto& m = up && glu ? c.glu : c.plain;
    const int cols = up ? F : N, k = up ? K : F;
    const double wgs = row_tiles(c.rows) * ((cols + m.bn - 1) / m.bn) / 256, nk = (k + 63) / 64;
    const double full = std::floor(wgs / m.at_once), rest = wgs - full * m.at_once;
    const double tiles = full * (nk * (m.step + m.more * (m.at_once - 1)) + m.begin) +
                         (rest > 0 ? nk * (m.step + m.more * (std::max(1.0, rest) - 1)) + m.begin : 0.0);
    return std::hypot(tiles, 2.0 * E * cols * k * (up && glu ? 2 : 1) / c.rate) + (double)P * (up ? 2.0 * F + 2.0 * K : 4.0 * N + 2.0 * F) / c.row_rate;
  };
  auto start = [&](const MoeCost& c) { return c.start + c.pair * P; };
  constexpr double by_rows = 1.12, by_ring = 1.08;
  double now = 0, best = 0;
  int best_ring = 0, now_ring = 0;
  for (int r : {64, 128, 256}) {
    if (r == 256 && !big) continue;
    double t, rule;  // of this form, and as the rule without the ring has it
    int on = 0;
    if (r == 64) {
      t = rule = start(kMoeCost[0]);
      const double extra = 0.5 * (start(kMoeCost[1]) - t);
      for (bool up : {true, false}) {
        const double a = us(kMoeCost[0], up), b = us(kMoeCost[1], up) + extra;
        const bool take = b * by_ring < a;
        rule += a, t += take ? b : a, on |= take ? (up ? 1 : 2) : 0;
      }
    } else {
      const MoeCost& c = kMoeCost[r == 128 ? 2 : 3];
      t = rule = start(c) + us(c, true) + us(c, false);
      on = r == 128 ? 3 : 0;
    }
    if (r == rows) now = rule, now_ring = on;
    if (best == 0 || t < best) best = t, *rows_out = r, best_ring = on;
  }
  *ring = best_ring;
  if (*rows_out != rows && best * by_rows >= now) *rows_out = rows, *ring = now_ring;
}

// act[r, f] = glu(h[order[r] / top] . gate_e[f], h[..] . up_e[f]) over the tile list (bf16), or gelu(h[..] . up_e[f])
// where there is no gate (wg null); tile_rows = the rows
// per tile the list was built with (moe_group): 64 or 128; use_ring: through the ring of k-steps where the operands allow it
void launch_moe_gate_up_tile(const void* h, int64_t ldh, const void* wg, const void* wu, const void* meta,
                             const void* order, void* act, int E, int maxt, int top, int F, int K, float limit,
                             float alpha, int tile_rows, const void* pw, int silu, int ilv, bool use_ring, hipStream_t st) {
  if (ilv && F % 16) throw std::runtime_error("moe_gate_up: gate and up in groups of 16 rows");
  if (tile_rows != 64 && tile_rows != 128) throw std::runtime_error("moe_gate_up: tile rows must be 64 or 128");
  if (maxt <= 0) return;
  if (maxt > 65535) throw std::runtime_error("moe_gate_up: too many row tiles");
  GemmTileArgs a{};
  a.A = (const bf16_t*)h; a.B = (const bf16_t*)wg; a.B2 = (const bf16_t*)wu; a.C = act;
  a.N = F; a.K = K; a.sAm = ldh; a.sBb = (int64_t)F * K; a.sBn = K; a.sCm = F;
  a.meta = (const int*)meta; a.order = (const int*)order; a.E = E; a.maxt = maxt; a.top = top;
  a.limit = limit; a.alpha = alpha; a.pw = (const float*)pw; a.silu = silu;
  if (ilv) {  // wg: [E, 2F, K]
    a.ilv = 1;
    a.B2 = a.B + (int64_t)16 * K;
    a.sBb = (int64_t)2 * F * K;
  }
  // 128-row tiles are 64 columns wide here: with two accumulator sets (gate and up) a 128x128 tile leaves one
  // workgroup per CU; at 128x64 two to three fit and hide each other's staging
  if (!wg) {
    a.B = (const bf16_t*)wu; a.B2 = nullptr;
    const bool ring = use_ring && moe_ring_ok(a, ldh, (int64_t)maxt * tile_rows / top, F);
    const int bn = tile_rows == 128 && F >= 512 ? 256 : tile_rows;
    dim3 g((F + bn - 1) / bn, maxt);
    if (ring && tile_rows == 128) tile_ring_kernel<GT_UP, bf16_t, 128, 128, 2><<<dim3((F + 127) / 128, maxt), 256, 0, st>>>(a);
    else if (ring) moe_ring64<GT_UP, bf16_t>(a, st);
    else if (bn == 256) gemm_tile_kernel<GT_UP, bf16_t, 128, 256><<<g, 256, 0, st>>>(a);
    else if (tile_rows == 128) gemm_tile_kernel<GT_UP, bf16_t, 128, 128><<<g, 256, 0, st>>>(a);
    else gemm_tile_kernel<GT_UP, bf16_t, 64, 64><<<g, 256, 0, st>>>(a);
    HIP_CHECK_LAUNCH();
    return;
  }
  dim3 g((F + 63) / 64, maxt);
  const bool ring = use_ring && moe_ring_ok(a, ldh, (int64_t)maxt * tile_rows / top, (int64_t)(ilv ? 2 : 1) * F);
  if (ring && tile_rows == 128) tile_ring_kernel<GT_GATE_UP, bf16_t, 128, 64, 2><<<g, 256, 0, st>>>(a);
  else if (ring) moe_ring64<GT_GATE_UP, bf16_t>(a, st);
  else if (tile_rows == 128) gemm_tile_kernel<GT_GATE_UP, bf16_t, 128, 64><<<g, 256, 0, st>>>(a);
  else gemm_tile_kernel<GT_GATE_UP, bf16_t, 64, 64><<<g, 256, 0, st>>>(a);
  HIP_CHECK_LAUNCH();
}

// y[r, n] = act[r, :] . down_e[n, :] over the tile list (fp32)
void launch_moe_down_tile(const void* act, const void* wd, const void* meta, void* y, int E, int maxt, int N, int F,
                          int tile_rows, bool use_ring, hipStream_t st) {
  if (tile_rows != 64 && tile_rows != 128) throw std::runtime_error("moe_down: tile rows must be 64 or 128");
  if (maxt <= 0) return;
  if (maxt > 65535) throw std::runtime_error("moe_down: too many row tiles");
  GemmTileArgs a{};
  a.A = (const bf16_t*)act; a.B = (const bf16_t*)wd; a.C = y;
  a.N = N; a.K = F; a.sAm = F; a.sBb = (int64_t)N * F; a.sBn = F; a.sCm = N;
  a.meta = (const int*)meta; a.E = E; a.maxt = maxt; a.top = 1;
  const int bn = tile_rows == 128 && N >= 512 ? 256 : tile_rows;
  dim3 g((N + bn - 1) / bn, maxt);
  const bool ring = use_ring && moe_ring_ok(a, F, (int64_t)maxt * tile_rows, N);
  if (ring && tile_rows == 128) tile_ring_kernel<GT_DOWN, float, 128, 128, 2><<<dim3((N + 127) / 128, maxt), 256, 0, st>>>(a);
  else if (ring) moe_ring64<GT_DOWN, float>(a, st);
  else if (bn == 256) gemm_tile_kernel<GT_DOWN, float, 128, 256><<<g, 256, 0, st>>>(a);
  else if (tile_rows == 128) gemm_tile_kernel<GT_DOWN, float, 128, 128><<<g, 256, 0, st>>>(a);
  else gemm_tile_kernel<GT_DOWN, float, 64, 64><<<g, 256, 0, st>>>(a);
  HIP_CHECK_LAUNCH();
}
