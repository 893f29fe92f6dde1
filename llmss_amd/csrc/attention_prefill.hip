// Causal variable-length flash-attention forward for prefill on MFMA (for
// S>1; reference materialises the [S,T] score matrix in fp32 with a CPU-built causal mask,
// gptj_modeling.py:128-169, gpt_bigcode_modeling.py:170-246).
//
// Layout: q/k/v are read straight from the fused QKV GEMM output [T, row_stride] (no
// split/permute copies, K9), sequences are packed back to back (cu_seqlens), GQA/MQA via
// kv_head = head / (nh / nkv). Output [T, nh*D] bf16 feeds the O-projection GEMM.
//
// Formulation ("swapped" products, guide §3 / T12 idea): per wave 16 query rows,
//   S^T[key][q] = K · Q^T          (A = K rows from LDS via ds_read_b128, B = Q^T in registers)
//   O^T[d][q]  += V^T · P^T        (A = V^T via ds_read_b64_tr_b16 transpose reads, B = P^T
//                                   taken straight from the S^T accumulators, no LDS trip)
// With S^T in the mfma_f32_16x16x32 C layout each lane owns ONE query row (lane & 15) and 16
// keys, so the online-softmax row max/sum is 15 in-register ops + 2 shuffles, and the P^T
// operand needs no data movement: the k-order permutation it implies is applied identically
// to the V^T operand through the addresses of the transpose reads.
// K/V tiles of 64 keys are register-staged into LDS rows padded by 32 B (conflict-free for
// both the b128 row reads and the tr_b16 column reads at D=128).
#include <type_traits>

#include "common.h"

constexpr float kLog2eP = 1.4426950408889634f;

template <int D>
__global__ __launch_bounds__(256) void attn_prefill_kernel(const bf16_t* __restrict__ qkv, int64_t row_stride,
                                                           const int* __restrict__ cu_seqlens, bf16_t* __restrict__ out,
                                                           int64_t out_stride, int nh, int nkv, int k_off, int v_off,
                                                           float scale_log2) {
  constexpr int BQ = 64, BKV = 64;
  constexpr int LD = D + 16;  // padded LDS row (elements)
  __shared__ __attribute__((aligned(16))) bf16_t Ks[BKV * LD];
  __shared__ __attribute__((aligned(16))) bf16_t Vs[BKV * LD];

  const int qb = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tok0 = cu_seqlens[b];
  const int len = cu_seqlens[b + 1] - tok0;
  if (qb * BQ >= len) return;
  const int kvh = h / (nh / nkv);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = lane & 15, g = lane >> 4;
  const int qrow = qb * BQ + w * 16 + li;  // this lane's query row within the sequence
  const bool qvalid = qrow < len;

  // Q^T fragments (B operand): lane holds Q[qrow][32ks + 8g .. +7]
  s16x8 qf[D / 32];
  {
    const bf16_t* qp = qkv + (int64_t)(tok0 + (qvalid ? qrow : len - 1)) * row_stride + (int64_t)h * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) qf[ks] = *reinterpret_cast<const s16x8*>(qp + 32 * ks);
  }
  f32x4 o[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -1.0e30f, lsum = 0.f;

  const int kv_end = min(len, qb * BQ + BQ);  // causal: keys < last query row of the block
  const int q_hi = qb * BQ + w * 16 + 15;     // last query row of this wave
  constexpr int CH = D / 8;                   // 16-B chunks per row
  for (int kv0 = 0; kv0 < kv_end; kv0 += BKV) {
    // ---- stage K, V tile (register staging) -----------------------------------------------
    __syncthreads();
#pragma unroll
    for (int c = threadIdx.x; c < BKV * CH; c += 256) {
      const int r = c / CH, ch = c % CH;
      const int kr = min(kv0 + r, len - 1);
      const bf16_t* src = qkv + (int64_t)(tok0 + kr) * row_stride + (int64_t)kvh * D + ch * 8;
      *reinterpret_cast<u16x8*>(&Ks[r * LD + ch * 8]) = *reinterpret_cast<const u16x8*>(src + k_off);
      *reinterpret_cast<u16x8*>(&Vs[r * LD + ch * 8]) = *reinterpret_cast<const u16x8*>(src + v_off);
    }
    __syncthreads();
    if (kv0 > q_hi) continue;  // whole tile is in this wave's causal future (keep barriers uniform)

    // ---- S^T = K Q^T : 4 key tiles of 16 ------------------------------------------------------
    f32x4 s[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks) {
        const s16x8 kf = *reinterpret_cast<const s16x8*>(&Ks[(kt * 16 + li) * LD + 32 * ks + 8 * g]);
        s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], s[kt], 0, 0, 0);
      }
    }
    // ---- mask + online softmax (lane owns query row qrow, keys kv0 + 16kt + 4g + i) ----------
    float mx = m;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kv0 + kt * 16 + 4 * g + i;
        float v = s[kt][i] * scale_log2;
        v = (key <= qrow) ? v : -1.0e30f;
        s[kt][i] = v;
        mx = fmaxf(mx, v);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float alpha = exp2f(m - mx);
    m = mx;
    float ps = 0.f;
    s16x8 pf[2];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = exp2f(s[kt][i] - mx);
        const bf16_t pb = f2bf(p);
        ps += bf2f(pb);
        pf[kt >> 1][(kt & 1) * 4 + i] = (short)pb;
      }
    ps += __shfl_xor(ps, 16, 64);
    ps += __shfl_xor(ps, 32, 64);
    lsum = lsum * alpha + ps;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) o[i] *= alpha;

    // ---- O^T += V^T P^T --------------------------------------------------------------------
    // transpose-read addresses: lane (4q + p) of its 16-lane group supplies row q, cols 4p..4p+3
    const int tq = li >> 2, tp = li & 3;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) {
        const bf16_t* a0 = &Vs[(32 * ks + 4 * g + tq) * LD + dt * 16 + 4 * tp];
        const bf16_t* a1 = a0 + 16 * LD;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(a0));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(a1));
        const s16x8 vf = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[ks], o[dt], 0, 0, 0);
      }
    }
  }
  if (!qvalid) return;
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  bf16_t* op = out + (int64_t)(tok0 + qrow) * out_stride + (int64_t)h * D + 4 * g;
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) {
    u16x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = f2bf(o[dt][i] * inv);
    *reinterpret_cast<u16x4*>(op + dt * 16) = r;
  }
}

// ------------------------------------------------------------------------------------------------
// v2: K/V tiles staged by LDS-DMA (buffer_load ... lds) into a two-slot ring, so tile j+1 streams in
// while tile j is computed (v1 above waits for register-staged loads before every tile); each wave
// owns QB 16-row query blocks, so every K / V fragment read from LDS feeds QB MFMAs; a workgroup
// serves GH query heads of one kv head (GQA: the K/V tile is loaded once for all of them); query
// blocks are dispatched last-first so the long causal rows start early.
// LDS rows are unpadded (DMA writes 1 KiB per wave-instruction linearly) with the 16-B chunk index
// XOR-swizzled by the row (swz below), applied on the source side of the DMA.
// FAST (v3): the same structure with a lighter softmax - the v2 loop issues ~2x more VALU than its 64
// MFMAs per tile can cover (MI355X_MICROARCH "vector-instruction ISSUE cost": 2 fillers per 16x16x32 gap):
//   * the causal / length mask only on tiles that cross the wave's diagonal or the sequence end;
//   * the row max on raw scores and the scale folded into the exponent (one fma per score);
//   * v_exp_f32 directly (no denormal range fix-ups: p < 2^-126 flushes to 0);
//   * deferred rescale (guide T13): the running max moves only when a row's max grows by more than 8
//     (log2 units), so p <= 2^8 and the O *= alpha sweep runs only when some row of the wave moved -
//     every l-side and o-side factor of a tile uses the same per-row alpha; whether one did is asked of the lanes' own scores, so
//     that a tile whose rows stand exchanges nothing between lanes (the sums meet at the end);
//   * the row sum accumulates the fp32 probabilities (v2 summed the bf16-rounded ones).
// us, the mask in a loop of its own, maxima by lane and eight sums of scores side by side, before and now: 3999 tokens, 32 heads of 128 232 ->
// 176 (158 with rows that are no multiple of 4 KB apart), two of 2048 tokens, 8 key heads 100 -> 82, four of 1000, 25 heads of 64 54 -> 42, two
// of 2000, 16 heads of 256 130 -> 112. A tile's scores beside the probabilities of the one before: 182; waves' priorities: 184.
// NW: waves per workgroup (4: two workgroups per CU; 8: one 512-thread workgroup per CU whose K/V tile
// feeds twice the query rows, halving the LDS-DMA traffic per FLOP).
template <int D, int QB, bool FAST, int NW = 4>
__global__ __launch_bounds__(64 * NW, 2) void attn_prefill_v2_kernel(const bf16_t* __restrict__ qkv, int64_t row_stride,
                                                                 int T, const int* __restrict__ cu_seqlens,
                                                                 bf16_t* __restrict__ out, int64_t out_stride, int nh,
                                                                 int nkv, int GH, int k_off, int v_off,
                                                                 float scale_log2, int nqb, int nseq) {
  constexpr int BKV = 64;
  constexpr int CH = D / 8;                    // 16-B chunks per row
  // LDS image swizzle of the 16-B chunk c of row r. D = 64 (128-B rows, two per bank row): c ^ (r & 7).
  // D >= 128 (rows span whole bank rows): c ^ ((r & 7) << 1) - conflict-free for both the b128 K reads
  // (16 rows x 1 chunk per lane group) and the b64 transpose reads of V, whose 32-lane groups take rows
  // r & 7 = 0..7 x two adjacent chunks: with c ^ (r & 15) those 32 lanes hit only 16 of the 32 8-B
  // bank slots (2-way conflicted: 33 % of LDS cycles, profiles/r3_prefill_attn PMC).
  auto swz = [](int c, int r) { return CH >= 16 ? c ^ ((r & 7) << 1) : c ^ (r & 7); };
  constexpr int TILE = BKV * D * 2;            // bytes of one K (or V) tile
  constexpr int RPI = 64 / CH;                 // rows per 1-KiB DMA wave-instruction
  constexpr int LPW = BKV / RPI / NW;          // DMA instructions per wave per tile (K and V each)
  static_assert(LPW >= 1, "tile / wave split");
  __shared__ __attribute__((aligned(16))) char smem[2 * 2 * TILE];  // [slot][K, V]

  const int G = nh / nkv;
  const int WPH = NW / GH;                     // waves per query head
  const int BQ = WPH * 16 * QB;
  // 1-D grid over (sequence, head group, query block). Workgroups are dealt round-robin to the 8 XCDs,
  // so consecutive ids share no L2: when the (sequence, head group) pairs split evenly over the XCDs,
  // every query block of one pair is sent to the same XCD (ids of one XCD = one residue mod 8) and
  // that pair's K/V is fetched into one L2 instead of eight. Within an XCD: heavy (late) blocks first.
  const int ngrp = G / GH;
  const int npair = nkv * ngrp * nseq;
  const int L = (int)blockIdx.x;
  int pair, qi_;
  if ((npair & 7) == 0) {
    const int slot = L >> 3;
    pair = (L & 7) + 8 * (slot / nqb);
    qi_ = slot % nqb;
  } else {
    pair = L / nqb;
    qi_ = L % nqb;
  }
  const int qb = nqb - 1 - qi_;
  const int b = pair / (nkv * ngrp);
  const int kvh = (pair % (nkv * ngrp)) / ngrp, grp = pair % ngrp;
  const int tok0 = cu_seqlens[b];
  const int len = cu_seqlens[b + 1] - tok0;
  const int q0 = qb * BQ;
  if (q0 >= len) return;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int h = kvh * G + grp * GH + w / WPH;
  const int wrow = q0 + (w % WPH) * 16 * QB;   // first query row of this wave

  // K / V descriptors from this sequence's first row; rows past the qkv tensor read as zero
  const uint64_t bytes = (uint64_t)(T - tok0) * (uint64_t)row_stride * 2;
  const uint32_t nrec = bytes > 0xFFFFFFF0ull ? 0xFFFFFFF0u : (uint32_t)bytes;
  const bf16_t* base = qkv + (int64_t)tok0 * row_stride + (int64_t)kvh * D;
  const auto rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base + k_off), (short)0, (int)nrec, 0x00020000);
  const auto rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base + v_off), (short)0, (int)nrec, 0x00020000);
  // per-lane (row, source-swizzled chunk) of the wave's first DMA instruction; instruction i is NW * RPI
  // rows further (a multiple of 8: same swizzle), added per issue - one live register instead of LPW
  static_assert((NW * RPI) % 8 == 0, "row step must keep the swizzle");
  const int r0_ = w * RPI + lane / CH;
  const uint32_t voff0 = (uint32_t)(r0_ * row_stride * 2 + (swz(lane % CH, r0_) << 4));
  // k position folded into the voffset (the range check covers voffset), soffset 0
#define PF_STAGE(J_)                                                                                           \
  do {                                                                                                         \
    char* sk_ = smem + ((J_) & 1) * 2 * TILE;                                                                  \
    const uint32_t kb_ = (uint32_t)((J_) * BKV) * (uint32_t)row_stride * 2u;                                   \
    _Pragma("unroll") for (int i_ = 0; i_ < LPW; ++i_) {                                                       \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (LDS_AS void*)(sk_ + (i_ * NW + w) * 1024), 16,             \
                                               voff0 + kb_ + (uint32_t)(i_ * NW * RPI * row_stride * 2), 0, 0, 0); \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (LDS_AS void*)(sk_ + TILE + (i_ * NW + w) * 1024), 16,      \
                                               voff0 + kb_ + (uint32_t)(i_ * NW * RPI * row_stride * 2), 0, 0, 0); \
    }                                                                                                          \
  } while (0)

  // Q^T fragments (B operand) of the wave's QB row blocks: lane holds Q[row][32ks + 8g .. +7]
  s16x8 qf[QB][D / 32];
#pragma unroll
  for (int qi = 0; qi < QB; ++qi) {
    const int r = min(wrow + qi * 16 + li, len - 1);
    const bf16_t* qp = qkv + (int64_t)(tok0 + r) * row_stride + (int64_t)h * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) qf[qi][ks] = *reinterpret_cast<const s16x8*>(qp + 32 * ks);
  }
  f32x4 o[QB][D / 16];
  float m[QB], lsum[QB];
#pragma unroll
  for (int qi = 0; qi < QB; ++qi) {
    m[qi] = -1.0e30f;
    lsum[qi] = 0.f;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) o[qi][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int kv_end = min(len, q0 + BQ);        // causal: no key past the block's last query row
  const int ntiles = (kv_end + BKV - 1) / BKV;
  const int w_hi = wrow + 16 * QB - 1;         // this wave's last query row
  const int tq = li >> 2, tp = li & 3;         // transpose-read lane roles (row q, 4 columns 4p..4p+3)
  PF_STAGE(0);
  // one tile of 64 keys; MASK: 0 none, 1 by position
  auto tile = [&](int j, auto mask_c) {
    constexpr bool MASK = decltype(mask_c)::value;
    const int kv0 = j * BKV;
    const char* Ks = smem + (j & 1) * 2 * TILE;
    const char* Vs = Ks + TILE;
    // ---- S^T = K Q^T: 4 key tiles of 16, each K fragment feeds QB MFMAs; 4 QB sums side by side ----
    f32x4 s[QB][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int qi = 0; qi < QB; ++qi) s[qi][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      s16x8 kf[4];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const int r = kt * 16 + li;
        kf[kt] = *reinterpret_cast<const s16x8*>(Ks + r * D * 2 + (swz(4 * ks + g, r) << 4));
      }
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int qi = 0; qi < QB; ++qi) s[qi][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kt], qf[qi][ks], s[qi][kt], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);  // (left alone, the last sums become chains of four behind one another)
    // ---- online softmax per row block (lane owns query row wrow + 16 qi + li) -------------
    s16x8 pf[QB][2];
    if constexpr (FAST) {
      float mx[QB];
      bool grew = false;
#pragma unroll
      for (int qi = 0; qi < QB; ++qi) {
        const int qrow = wrow + qi * 16 + li;
        mx[qi] = -1.0e30f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if constexpr (MASK) {
              const int key = kv0 + kt * 16 + 4 * g + i;
              s[qi][kt][i] = (key <= qrow && key < len) ? s[qi][kt][i] : -1.0e30f;
            }
            mx[qi] = fmaxf(mx[qi], s[qi][kt][i]);
          }
        mx[qi] *= scale_log2;
        grew |= mx[qi] > m[qi] + 8.f;
      }
      if (__ballot(grew)) {  // some row's maximum moves: lanes of a row agree on it only here
#pragma unroll
        for (int qi = 0; qi < QB; ++qi) {
          const float rmx = xor32_max(xor16_max(mx[qi]));
          const bool resc = rmx > m[qi] + 8.f;
          const float alpha = resc ? __builtin_amdgcn_exp2f(m[qi] - rmx) : 1.f;
          if (resc) m[qi] = rmx;
          lsum[qi] *= alpha;
#pragma unroll
          for (int i = 0; i < D / 16; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[qi][i][e] *= alpha;
        }
      }
#pragma unroll
      for (int qi = 0; qi < QB; ++qi) {
        const float nm = -m[qi];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = __builtin_amdgcn_exp2f(fmaf(s[qi][kt][i], scale_log2, nm));
            lsum[qi] += p;
            pf[qi][kt >> 1][(kt & 1) * 4 + i] = (short)f2bf(p);
          }
      }
    } else {
#pragma unroll
    for (int qi = 0; qi < QB; ++qi) {
      const int qrow = wrow + qi * 16 + li;
      float mx = m[qi];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = kv0 + kt * 16 + 4 * g + i;
          float v = s[qi][kt][i] * scale_log2;
          v = (key <= qrow && key < len) ? v : -1.0e30f;
          s[qi][kt][i] = v;
          mx = fmaxf(mx, v);
        }
      mx = xor32_max(xor16_max(mx));
      const float alpha = exp2f(m[qi] - mx);
      m[qi] = mx;
      float ps = 0.f;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bf16_t pb = f2bf(exp2f(s[qi][kt][i] - mx));
          ps += bf2f(pb);
          pf[qi][kt >> 1][(kt & 1) * 4 + i] = (short)pb;
        }
      ps = xor32_sum(xor16_sum(ps));
      lsum[qi] = lsum[qi] * alpha + ps;
#pragma unroll
      for (int i = 0; i < D / 16; ++i) o[qi][i] *= alpha;
    }
    }
    // ---- O^T += V^T P^T (V^T by transpose reads of the swizzled V tile), each V fragment feeds QB MFMAs
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int r0 = 32 * ks + 4 * g + tq, r1 = r0 + 16;
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) {
        const int c = 2 * dt + (tp >> 1);
        const char* a0 = Vs + r0 * D * 2 + (swz(c, r0) << 4) + (tp & 1) * 8;
        const char* a1 = Vs + r1 * D * 2 + (swz(c, r1) << 4) + (tp & 1) * 8;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(a0));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(a1));
        const s16x8 vf = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
#pragma unroll
        for (int qi = 0; qi < QB; ++qi) o[qi][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[qi][ks], o[qi][dt], 0, 0, 0);
      }
    }
  };
  // tiles that no mask touches first; the last ones, on the wave's diagonal or the sequence's end, in a loop of their own (the positions'
  // arithmetic beside the other, though skipped, was a sixth of its vector instructions)
  const int whole = FAST ? min(min((wrow + 1) / BKV, len / BKV), ntiles) : 0;
  int j = 0;
#define PF_NEXT()                                                                            \
  do {                                                                                       \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                         \
    __builtin_amdgcn_s_barrier(); /* tile j landed for every wave; slot (j+1)&1 is free */   \
    asm volatile("" ::: "memory");                                                           \
    if (j + 1 < ntiles) PF_STAGE(j + 1);                                                     \
  } while (0)
  for (; j < whole; ++j) {
    PF_NEXT();
    tile(j, std::false_type{});
  }
  for (; j < ntiles; ++j) {
    PF_NEXT();
    if (j * BKV > w_hi) continue;              // the whole tile is in this wave's causal future
    tile(j, std::true_type{});
  }
  if constexpr (FAST) {  // (the row sums, so far by lane)
#pragma unroll
    for (int qi = 0; qi < QB; ++qi) lsum[qi] = xor32_sum(xor16_sum(lsum[qi]));
  }
#undef PF_NEXT
#undef PF_STAGE
#pragma unroll
  for (int qi = 0; qi < QB; ++qi) {
    const int qrow = wrow + qi * 16 + li;
    if (qrow >= len) continue;
    const float inv = lsum[qi] > 0.f ? 1.f / lsum[qi] : 0.f;
    bf16_t* op = out + (int64_t)(tok0 + qrow) * out_stride + (int64_t)h * D + 4 * g;
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
      u16x4 r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = f2bf(o[qi][dt][i] * inv);
      *reinterpret_cast<u16x4*>(op + dt * 16) = r;
    }
  }
}

// version 3 (default): v2 with the light softmax; waves per workgroup 0 = auto (8 for D = 256, else 4)
static int g_prefill_version = 3;
static int g_prefill_nw = 0;
void attn_prefill_set_waves(int nw) { g_prefill_nw = (nw == 4 || nw == 8) ? nw : 0; }
void attn_prefill_set_version(int v) { g_prefill_version = (v >= 1 && v <= 3) ? v : 3; }

void launch_attn_prefill(const void* qkv, int64_t row_stride, int T, const void* cu_seqlens, void* out,
                         int64_t out_stride, int B, int max_seqlen, int nh, int nkv, int D, int k_off, int v_off,
                         float scale, hipStream_t st) {
  if (nh % nkv) throw std::runtime_error("attn_prefill: nh must be a multiple of nkv");
  if (B == 0 || max_seqlen == 0) return;
  auto Q = (const bf16_t*)qkv;
  auto CU = (const int*)cu_seqlens;
  auto O = (bf16_t*)out;
  const float sl = scale * kLog2eP;
  // v3 by default (profiles/r3_prefill_attn, bench/attn_prefill_bench.py: faster than v1 and v2 on every
  // measured config); v2 keeps its dispatch (v1 for D = 256 and D = 64 beyond 2K tokens)
  const bool fast = g_prefill_version == 3;
  if (fast || (g_prefill_version == 2 && D != 256 && !(D == 64 && max_seqlen > 2048))) {
    if (row_stride % 8 || k_off % 8 || v_off % 8)
      throw std::runtime_error("attn_prefill: 16-B aligned rows and k/v offsets required");
    if ((uint64_t)64 * row_stride * 2 >= (1ull << 31)) throw std::runtime_error("attn_prefill: row stride too large");
    const int G = nh / nkv;
    const int NW = !fast ? 4 : (g_prefill_nw ? g_prefill_nw : (D == 256 ? 8 : 4));
    const int GH = (NW == 8 && G % 8 == 0) ? 8 : (G % 4 == 0 ? 4 : (G % 2 == 0 ? 2 : 1));
    const int QB = D == 256 ? 1 : 2;  // D = 256: one row block per wave keeps O + Q in the register budget
    const int BQ = (NW / GH) * 16 * QB;
    const int nqb = (max_seqlen + BQ - 1) / BQ;
    dim3 grid(nqb * nkv * (G / GH) * B);
    const int key = (D * 2 + (fast ? 1 : 0)) * 16 + NW;
    switch (key) {
      case 128 * 16 + 4: attn_prefill_v2_kernel<64, 2, false><<<grid, 256, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 129 * 16 + 4: attn_prefill_v2_kernel<64, 2, true><<<grid, 256, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 129 * 16 + 8: attn_prefill_v2_kernel<64, 2, true, 8><<<grid, 512, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 256 * 16 + 4: attn_prefill_v2_kernel<128, 2, false><<<grid, 256, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 257 * 16 + 4: attn_prefill_v2_kernel<128, 2, true><<<grid, 256, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 257 * 16 + 8: attn_prefill_v2_kernel<128, 2, true, 8><<<grid, 512, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 513 * 16 + 4: attn_prefill_v2_kernel<256, 1, true><<<grid, 256, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      case 513 * 16 + 8: attn_prefill_v2_kernel<256, 1, true, 8><<<grid, 512, 0, st>>>(Q, row_stride, T, CU, O, out_stride, nh, nkv, GH, k_off, v_off, sl, nqb, B); break;
      default: throw std::runtime_error("attn_prefill: head_dim must be 64, 128 or 256");
    }
    HIP_CHECK_LAUNCH();
    return;
  }
  dim3 grid((max_seqlen + 63) / 64, nh, B);
  switch (D) {
    case 64: attn_prefill_kernel<64><<<grid, 256, 0, st>>>(Q, row_stride, CU, O, out_stride, nh, nkv, k_off, v_off, sl); break;
    case 128: attn_prefill_kernel<128><<<grid, 256, 0, st>>>(Q, row_stride, CU, O, out_stride, nh, nkv, k_off, v_off, sl); break;
    case 256: attn_prefill_kernel<256><<<grid, 256, 0, st>>>(Q, row_stride, CU, O, out_stride, nh, nkv, k_off, v_off, sl); break;
    default: throw std::runtime_error("attn_prefill: head_dim must be 64, 128 or 256");
  }
  HIP_CHECK_LAUNCH();
}
