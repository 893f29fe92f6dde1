// Softmax attention with a sink, a soft cap and head mixing in one kernel (attention_sink.hip's talk form, bf16 pages): the weights
// of all heads are mixed before they meet the values, so that a head's sum runs over its own group's values only.
//
//   s_h(i, j) = cap * tanh(scale * q_h(i) . k_g(j) / cap)     p_h(i, j) = exp(s_h(i, j)) / L_h(i),  L_h(i) = 1 + sum_j exp(s_h(i, j))
//   y_h(i) = c * sum_j (sum_h' talk[h, h'] p_h'(i, j)) v_g(h)(j)
//
// Mixing before the values needs the denominators first: the keys are walked twice, once for L and once for the weighted sums. The
// cap bounds every score, so exp needs no running maximum: the host takes this path for caps up to 60 (exp below 2^87, and 2^127 holds
// 10^12 keys of it). The form that mixes afterwards (attention_sink.hip, then talk_mix) does G times the products with the values,
// in column chunks of 256 that each score again, and leaves an fp32 [T, H, G * vdim] in memory.
//
// A workgroup serves 16 rows of a sequence and all heads, 32 keys at a time; wave (group, half) owns two of the group's four heads:
//   S^T[key][row] = K . Q^T   (A = 16 keys from LDS, B = Q^T in registers: a lane owns row li, keys 4 g + i)
//   its fp32 weights go to LDS, from where every wave takes all heads' weights of four keys and mixes them on the fp32 matrix
//   instructions, W[head][row] = talk . P[head'][row] a key; the mixed weights return through LDS as bf16 operands of
//   O^T[c][row] += V^T . W^T  (A = V^T by transposing LDS reads of the group's 32 keys).
// Two barriers per 32 keys; the next keys' scores and weights stand beside this tile's products with the values.
// A CU gets about 36 KB a microsecond from the L2, and 16 rows meet 2 or 3 KB a key: so keys and values are read once a workgroup,
// whole rows (all groups' keys side by side) an instruction, into registers a tile ahead and then to LDS. Operands straight from
// the cache, each wave its own 64-byte pieces, took 5.3 us per 32 keys of both walks at 16 heads, this 3.5: about half of it the vector
// ALUs (3 transcendental instructions a pair of row and key and head in either walk), the rest barriers and waits for LDS.
// us, the two kernels of attention_sink.hip and this: 16 heads of 128, 8 prompts of 1024 418 and 153, 64 of 24 47 and 17, one of 4000 442 and
// 429; 8 heads 112 and 95, 23 and 10, 168 and 302. One workgroup walks all keys of its rows, where the other form spreads groups and
// column chunks over workgroups: while those still fit the chip it is the faster one (2 portions of 512 behind 1500 keys: 104 and 174,
// one row behind 4000: 149 and 438), which is what the caller's rule weighs. Two and four groups only: 32 keys and values of eight, with their 32
// heads' weights in fp32 and mixed, would take 224 KB of LDS.
#include "anytype.h"

namespace {

struct MixAttnArgs {
  const float* q;  // [T, H * DK]
  const bf16_t *kc, *vc;
  const int* bt;
  const int *cu, *ctx;
  const float* talk;  // [H, H]
  bf16_t* y;
  int64_t ldy;
  int maxb, bs, bshift;
  float scale, cap, c;
};

constexpr int kMixPages = 1024;  // page ids of a sequence, held in LDS

}  // namespace

template <int DK, int NG>
__global__ __launch_bounds__(128 * NG, 2) void mix_attn_kernel(MixAttnArgs p) {
  constexpr int H = 4 * NG, KS = DK / 32, VD = 128, NVT = VD / 16, NW = 2 * NG;
  constexpr int KB = DK * 2, VB = VD * 2;      // bytes of a group's key, of its value
  constexpr int KT = 32 * KB, VT = 32 * VB;    // of their tiles
  constexpr int CK = NG * DK / 8, CV = NG * VD / 8;  // 16-byte chunks of a cached row
  constexpr int NK = 32 * CK / (64 * NW), NV = 32 * CV / (64 * NW);  // that a lane moves per tile
  __shared__ __attribute__((aligned(16))) char Ks[NG * KT];
  __shared__ __attribute__((aligned(16))) char Vs[NG * VT];
  __shared__ __attribute__((aligned(16))) f32x4 Ps[H][2][64];  // fp32 weights: head, half of the tile, lane (row, four keys)
  __shared__ __attribute__((aligned(16))) u16x8 Ws[H][64];     // mixed: head, lane (row, four keys of each half)
  __shared__ int pages[kMixPages];
  int bx, by, b;
  causal_block_order(bx, by, b);
  const int t0 = p.cu[b], qlen = p.cu[b + 1] - t0, r0 = bx * 16;
  if (r0 >= qlen) return;
  const int p0 = p.ctx[b] - qlen;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4, grp = w >> 1, h0 = grp * 4 + (w & 1) * 2;
  const int total = min(p0 + min(qlen, r0 + 16), p.maxb << p.bshift);  // keys that the last row sees
  const int qpos = p0 + min(r0 + li, qlen - 1), first = p0 + r0;
  if (total <= 0) {  // a padded row has no keys
    for (int i = threadIdx.x; i < (qlen - r0) * H * VD && i < 16 * H * VD; i += blockDim.x)
      p.y[(int64_t)(t0 + r0 + i / (H * VD)) * p.ldy + i % (H * VD)] = 0;
    return;
  }
  const int* bt = p.bt + (int64_t)b * p.maxb;
  const int npages = (total + p.bs - 1) >> p.bshift;
  for (int i = threadIdx.x; i < npages; i += blockDim.x) pages[i] = bt[i];
  s16x8 qf[2][KS];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const float* qp = p.q + ((int64_t)(t0 + min(r0 + li, qlen - 1)) * H + h0 + n) * DK + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(qp + 32 * ks), c = *reinterpret_cast<const f32x4*>(qp + 32 * ks + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) qf[n][ks][j] = (short)f2bf(a[j]), qf[n][ks][4 + j] = (short)f2bf(c[j]);
    }
  }
  float tk[H / 4];  // talk [target li][head 4 s + g]: the mixing products' A operand
#pragma unroll
  for (int i = 0; i < H / 4; ++i) tk[i] = li < H ? p.talk[li * H + 4 * i + g] : 0.f;
  __syncthreads();
  auto barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // (one path: a load behind a branch would make each of these wait for the one before)
  auto slot_of = [&](int key) { return ((int64_t)pages[key >> p.bshift] << p.bshift) + (key & (p.bs - 1)); };
  // 32 keys' or values' rows from u0 on: chunk c of a row is group c / (chunks of a group)'s
  u16x8 kr[NK], vr[NV];
  auto fetch_k = [&](int u0) {
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int at = threadIdx.x + j * 64 * NW, r = at / CK, c = at % CK;
      kr[j] = *reinterpret_cast<const u16x8*>(p.kc + slot_of(min(u0 + r, total - 1)) * (NG * DK) + c * 8);
    }
  };
  auto fetch_v = [&](int u0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int at = threadIdx.x + j * 64 * NW, r = at / CV, c = at % CV;
      vr[j] = *reinterpret_cast<const u16x8*>(p.vc + slot_of(min(u0 + r, total - 1)) * (NG * VD) + c * 8);
    }
  };
  // LDS places: a group's tile is rows of KB or VB bytes; chunk c of key row r lies at c ^ (r & 15 or 7), so that 16 keys' operand
  // chunks meet every bank once, a value row's 32-byte block d at d ^ (r & 7), so that a transposing read of 16 rows meets every bank twice
  constexpr int KX = DK / 8 - 1;
  auto store_k = [&](char* ks) {
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int at = threadIdx.x + j * 64 * NW, r = at / CK, c = at % CK, gi = c / (DK / 8), cc = c % (DK / 8);
      *reinterpret_cast<u16x8*>(ks + gi * KT + r * KB + ((cc ^ (r & KX)) << 4)) = kr[j];
    }
  };
  auto store_v = [&] {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int at = threadIdx.x + j * 64 * NW, r = at / CV, c = at % CV, gi = c / (VD / 8), cc = c % (VD / 8);
      *reinterpret_cast<u16x8*>(Vs + gi * VT + r * VB + ((cc ^ ((r & 7) << 1)) << 4)) = vr[j];
    }
  };
  // raw scores of the tile's 32 keys: lane (row li), keys 16 kt + 4 g + i, heads h0, h0 + 1
  auto scores = [&](const char* ks, f32x4(&s)[2][2]) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int n = 0; n < 2; ++n) s[kt][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const s16x8 kf = *reinterpret_cast<const s16x8*>(ks + grp * KT + (16 * kt + li) * KB + (((4 * q + g) ^ (li & KX)) << 4));
#pragma unroll
        for (int n = 0; n < 2; ++n) s[kt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[n][q], s[kt][n], 0, 0, 0);
      }
    }
  };
  constexpr float kLog2e = 1.4426950408889634f;
  const float capx = 2.0f * kLog2e * p.scale / p.cap, capy = -2.0f * p.cap * kLog2e;
  // exp2 of (the capped score * log2 e + off): tanh(x) = 1 - 2 / (exp(2 x) + 1). Keys that a row does not see weigh nothing.
  auto weigh = [&](int u0, const float(&off)[2], f32x4(&s)[2][2]) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[kt][n][i] = __builtin_amdgcn_exp2f(fmaf(capy, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(s[kt][n][i] * capx) + 1.0f), off[n]));
    if (u0 + 31 > first) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[kt][n][i] = u0 + 16 * kt + 4 * g + i <= qpos ? s[kt][n][i] : 0.f;
    }
  };

  // ---- first walk: the denominators of (row li, heads h0, h0 + 1); tiles in Ks and Vs by turns
  const float off0 = -0.5f * capy;
  float off[2] = {off0, off0};
  {
    f32x4 sum[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    fetch_k(0);
    for (int u0 = 0; u0 < total; u0 += 32) {
      char* ks = u0 & 32 ? Vs : Ks;
      store_k(ks);
      fetch_k(u0 + 32 < total ? u0 + 32 : 0);  // (behind the last one the second walk's first)
      barrier();
      f32x4 s[2][2];
      scores(ks, s);
      weigh(u0, off, s);
#pragma unroll
      for (int n = 0; n < 2; ++n) sum[n] += s[0][n] + s[1][n];
    }
#pragma unroll
    for (int n = 0; n < 2; ++n)  // (log2)
      off[n] = off0 - __builtin_amdgcn_logf(1.0f + xor32_sum(xor16_sum((sum[n][0] + sum[n][1]) + (sum[n][2] + sum[n][3]))));
  }

  // ---- second walk
  f32x4 o[2][NVT];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int i = 0; i < NVT; ++i) o[n][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto publish = [&](int u0) {  // the weights of 32 keys from u0 on
    f32x4 s[2][2];
    scores(Ks, s);
    weigh(u0, off, s);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int n = 0; n < 2; ++n) Ps[h0 + n][kt][lane] = s[kt][n];
  };
  constexpr int QW = 8 / NW;  // key quads of a tile that a wave mixes
  const int tq = li >> 2, tp = li & 3, vrow = 4 * g + tq;  // (16 rows further on the low three bits are the same)
  barrier();  // every wave is done with the first walk's tiles
  store_k(Ks);
  fetch_k(32);
  fetch_v(0);
  barrier();
  publish(0);
  for (int u0 = 0; u0 < total; u0 += 32) {
    barrier();  // the weights are there; every wave is done with the keys, and with the values of the tile before
    store_k(Ks);
    store_v();
    fetch_k(u0 + 64);
    fetch_v(u0 + 32);
#pragma unroll
    for (int q = 0; q < QW; ++q) {
      const int quad = w * QW + q, kt = quad >> 2, at = li + 16 * (quad & 3);  // keys 16 kt + 4 (quad & 3) ..
      f32x4 m[4];  // per key: targets 4 g .. 4 g + 3 of row li
#pragma unroll
      for (int j = 0; j < 4; ++j) m[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < H / 4; ++i) {
        const f32x4 e = Ps[4 * i + g][kt][at];
#pragma unroll
        for (int j = 0; j < 4; ++j) m[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(tk[i], e[j], m[j], 0, 0, 0);
      }
      if (H == 16 || g < 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          reinterpret_cast<u16x4*>(&Ws[4 * g + i][at])[kt] = u16x4{f2bf(m[0][i]), f2bf(m[1][i]), f2bf(m[2][i]), f2bf(m[3][i])};
      }
    }
    barrier();
    s16x8 pf[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) pf[n] = __builtin_bit_cast(s16x8, Ws[h0 + n][lane]);
    const char* vs = Vs + grp * VT + vrow * VB + tp * 8;
#pragma unroll
    for (int dt = 0; dt < NVT; ++dt) {
      const char* a0 = vs + ((dt ^ (vrow & 7)) << 5);
      const s16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(a0));
      const s16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(a0 + 16 * VB));
      const s16x8 vf = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
      for (int n = 0; n < 2; ++n) o[n][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[n], o[n][dt], 0, 0, 0);
    }
    publish(u0 + 32);  // (behind the last tile: weights of zero, not read)
  }
  if (r0 + li >= qlen) return;
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    bf16_t* yp = p.y + (int64_t)(t0 + r0 + li) * p.ldy + (h0 + n) * VD + 4 * g;
#pragma unroll
    for (int dt = 0; dt < NVT; ++dt) {
      const f32x4 v = o[n][dt] * p.c;
      *reinterpret_cast<u16x4*>(yp + dt * 16) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
    }
  }
}

// Shapes that the kernel takes (the pages in bf16, rows of 16-byte alignment, and y's of 8 bytes are the caller's to check): pages of a
// power of two, found by a shift, as many as LDS holds
bool mix_attn_ok(int H, int G, int dim, int vdim, int bs, int maxb, float cap) {
  return (G == 2 || G == 4) && H == 4 * G && (dim == 64 || dim == 128) && vdim == 128 && bs > 0 && (bs & (bs - 1)) == 0 &&
         maxb <= kMixPages && cap > 0.f && cap <= 60.f;
}

// y [T, H * vdim] (bf16, row stride ldy) of B sequences' portions of at most max_qlen rows; q fp32 [T, H * dim]
void launch_mix_attn(const void* q, const void* kc, const void* vc, const void* bt, int maxb, const void* cu, const void* ctx,
                     const void* talk, float c, void* y, int64_t ldy, int B, int max_qlen, int H, int G, int dim, int vdim, int bs,
                     float scale, float cap, hipStream_t st) {
  if (B == 0 || max_qlen <= 0) return;
  if (!mix_attn_ok(H, G, dim, vdim, bs, maxb, cap)) throw std::runtime_error("mixed attention: shape not built");
  if (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) & 15 || (uintptr_t)y & 7 || ldy % 4)
    throw std::runtime_error("mixed attention: alignment");
  if (B > 65535) throw std::runtime_error("mixed attention: too many sequences");
  MixAttnArgs a{(const float*)q, (const bf16_t*)kc, (const bf16_t*)vc, (const int*)bt, (const int*)cu, (const int*)ctx,
                (const float*)talk, (bf16_t*)y, ldy, maxb, bs, __builtin_ctz(bs), scale, cap, c};
  dim3 grid((max_qlen + 15) / 16, 1, B);
#define MIX(DK_, NG_) mix_attn_kernel<DK_, NG_><<<grid, 128 * NG_, 0, st>>>(a)
  if (dim == 64) {
    if (G == 2) MIX(64, 2);
    else MIX(64, 4);
  } else if (G == 2) MIX(128, 2);
  else MIX(128, 4);
#undef MIX
  HIP_CHECK_LAUNCH();
}
