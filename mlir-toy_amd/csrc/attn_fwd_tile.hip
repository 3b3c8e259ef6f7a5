// attn_fwd_tile.hip — head_dim-64, 16-bit HTile attention forward for gfx950.
//
// Semantics are those of attn_fwd.hip. The structure is that of the
// head_dim-128 kernel (attn_fwd_d128.hip): 256 threads = 4 waves, 128 query
// rows (32 per wave), 64-key blocks, K and V tiles HBM -> LDS by
// global_load_lds_dwordx4 into two slots per operand, the transposed products
//   S^T = K . Q^T   (A = K rows from LDS, B = Q^T in VGPRs)
//   O^T = V^T . P^T (A = V^T from LDS via ds_read_b64_tr_b16, B = P^T)
// on v_mfma_f32_32x32x16 (one query row per lane), block j+1's QK^T in the
// MFMA stream of block j's P.V, and the lazily moved running max.
//
// Bound: at head_dim 64 a key block's softmax (128 vector instructions a
// wave, about 640 cycles) outweighs its 16 MFMAs (512 cycles); counters show
// the two units busy in 87% of the cycles, half of the matrix time under
// vector work. Two work-groups per CU (182 registers). Three or four of them
// (127 registers, with the copies' rare tail computed in place) measured the
// same within 3%, and a barrier for every second key block (four slots per
// operand) 8% slower, so neither occupancy nor the barrier holds it back.
// Measured (GPU time, against a kernel that staged K and V through registers
// and transposed V while writing it to LDS): B4 H16 S2048 causal 58.5 -> 43-45
// us (770 TFLOP/s), without the mask 105 -> 73-75 us (930), B1 H8 S4096 causal
// 83 -> 52 us, B4 H8 S55 5.1 -> 4.0 us.
#include "attn_args.h"
#include "attn_tile.h"
#include "kernels.h"

namespace neptune {
namespace {

template <class E, int HD, bool CAUSAL>
__global__ __launch_bounds__(NT, 2) void attn_fwd_tile(AttnArgs a) {
  typedef typename E::vec8 V8;
  constexpr int TILE = TileLoader<HD>::TILE_BYTES;
  constexpr int ROWB = HD * 2;   // bytes per LDS row
  constexpr int NST = HD / 16;   // QK^T k-steps
  constexpr int NB = HD / 32;    // 32-wide head_dim blocks of O^T
  constexpr int NQK = 2 * NST, NPV = 4 * NB;  // MFMAs per key block
  // K slots 0 and 1, then V slots 0 and 1; block t uses slot t & 1
  __shared__ __attribute__((aligned(16))) uint8_t smem[4 * TILE];
  const uint8_t *const kt0 = smem;
  const uint8_t *const vt0 = smem + 2 * TILE;
  auto kslot = [&](int t) { return kt0 + (t & 1) * TILE; };
  auto vslot = [&](int t) { return vt0 + (t & 1) * TILE; };

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, g = lane >> 5;

  // Work-group -> (kv head, query head of its group, query block): kv heads
  // fastest, so that (with a multiple of 8 of them) id % 8, the XCD, fixes
  // the kv head modulo 8 and all readers of a head's K and V share an L2;
  // the heaviest causal query blocks first
  const int BHk = a.BH / a.group;
  const int id = blockIdx.x;
  const int bhk = __builtin_amdgcn_readfirstlane(id % BHk);
  const int rest = id / BHk;
  const int qb = __builtin_amdgcn_readfirstlane(a.nqb - 1 - rest / a.group);
  const int Hk = a.Hq / a.group;
  const int b = __builtin_amdgcn_readfirstlane(bhk / Hk);
  const int hk = bhk - b * Hk;
  const int h = __builtin_amdgcn_readfirstlane(hk * a.group + rest % a.group);
  const uint16_t *qp = (const uint16_t *)a.q + b * a.qs0 + h * a.qs1;
  const uint16_t *kp = (const uint16_t *)a.k + b * a.ks0 + hk * a.ks1;
  const uint16_t *vp = (const uint16_t *)a.v + b * a.vs0 + hk * a.vs1;

  const int row0 = qb * BM + w * 32, row = row0 + lq;
  // key blocks of the work-group and of this wave
  int nv = (a.Sk + BN - 1) / BN, nkw = nv;
  if (CAUSAL) {
    const int last_wg = qb * BM + BM - 1 + a.off, last_w = row0 + 31 + a.off;
    nv = min(nv, last_wg < 0 ? 0 : last_wg / BN + 1);
    nkw = min(nv, last_w < 0 ? 0 : last_w / BN + 1);
  }

  const TileLoader<HD> kl = make_loader<HD, false>(kp, a.ks2, w, lane);
  const TileLoader<HD> vl = make_loader<HD, true>(vp, a.vs2, w, lane);
  auto load_k = [&](int t) { tile_to_lds<false>(kl, t * BN, a.Sk, kslot(t), w); };
  auto load_v = [&](int t) { tile_to_lds<true>(vl, t * BN, a.Sk, vslot(t), w); };
  if (nv > 0) load_k(0);
  if (nv > 1) load_k(1);
  if (nv > 0) load_v(0);

  // Q^T operand: k-step st covers head_dim 16 st + 8 g .. +7 of the row
  u32x4 qf[NST];
#pragma unroll
  for (int st = 0; st < NST; ++st)
    qf[st] = row < a.Sq ? *(const u32x4 *)(qp + row * a.qs2 + 16 * st + 8 * g)
                        : u32x4{0, 0, 0, 0};

  // per-lane LDS byte offsets of the operand reads
  int ka[NST];  // K: row lq (+32 kb), logical unit 2 st + g
#pragma unroll
  for (int st = 0; st < NST; ++st)
    ka[st] = lq * ROWB + (((2 * st + g) ^ tile_swizzle<HD, false>(lq)) << 4);
  int va[NB];  // V^T: transpose read, rows 4 g + i (+16 c + 8 t), columns 32 nb + 16 dh + 4 q
  {
    const int s16 = lane & 15, i = s16 >> 2, q = s16 & 3, dh = (lane >> 4) & 1;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      va[nb] = (4 * g + i) * ROWB + (((4 * nb + 2 * dh) ^ tile_swizzle<HD, true>(i)) << 4) + 8 * q;
  }

  f32x16 o[NB];
  f32x16 s[2];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[nb][r] = 0.0f;
  float m = kNegFltMax, lsum = 0.0f;
  const float sc = a.scale2;
  const f32x16 zero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

  // The A operand of MFMA i = 2 st + kb of S^T = K.Q^T (32 keys x 16 head_dim)
  auto k_operand = [&](const uint8_t *kt, int i) {
    return *(const u32x4 *)(kt + (i & 1) * 32 * ROWB + ka[i >> 1]);
  };
  // S^T of one key block, its first two A operands already read (k0, k1)
  auto qk_from = [&](const uint8_t *kt, const u32x4 &k0, const u32x4 &k1) {
#pragma unroll
    for (int i = 0; i < NQK; ++i) {
      const u32x4 A = i == 0 ? k0 : i == 1 ? k1 : k_operand(kt, i);
      s[i & 1] = E::mfma32(as_vec8<V8>(A), as_vec8<V8>(qf[i >> 1]), i < 2 ? zero16 : s[i & 1]);
    }
    // the remaining operand reads run two MFMAs ahead
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
#pragma unroll
    for (int i = 0; i < NQK - 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
  };
  // The A operand of P.V step st (V^T: head_dim rows 32 nb .., keys 16 c ..)
  auto v_operand = [&](const uint8_t *vt, int st) {
    const int c = st / NB, nb = st % NB;
    const u32x2 a0 = __builtin_bit_cast(u32x2, lds_read_tr16(vt + 16 * c * ROWB + va[nb]));
    const u32x2 a1 = __builtin_bit_cast(u32x2, lds_read_tr16(vt + (16 * c + 8) * ROWB + va[nb]));
    return u32x4{a0[0], a0[1], a1[0], a1[1]};
  };

  wait_vmem();
  __syncthreads();
  if (nkw > 0) qk_from(kslot(0), k_operand(kslot(0), 0), k_operand(kslot(0), 1));
  __syncthreads();  // every wave is done with K slot 0 before it is refilled

  for (int jb = 0; jb < nv; ++jb) {
    // K of block jb + 2 goes to the slot block jb's K has left, V of block
    // jb + 1 to the slot of block jb - 1's V
    if (jb + 2 < nv) load_k(jb + 2);
    if (jb + 1 < nv) load_v(jb + 1);
    if (jb < nkw) {
      // the first two V^T operands of this block's P.V, read before the softmax
      const uint8_t *vt = vslot(jb);
      const u32x4 vp0 = v_operand(vt, 0), vp1 = v_operand(vt, 1);
      const int key0 = jb * BN;
      if ((key0 + BN > a.Sk) || (CAUSAL && key0 + BN - 1 > row0 + a.off)) {
        // element (kb, r) holds key key0 + 4 g + c with c = 32 kb + 8 (r >> 2)
        // + (r & 3): it is masked when c passes the lane's last visible key
        int lim = a.Sk - 1 - key0 - 4 * g;
        if (CAUSAL) lim = min(lim, row + a.off - key0 - 4 * g);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * kb + 8 * (r >> 2) + (r & 3) > lim) s[kb][r] = -INFINITY;
      }
      // p = 2^(s sc - m) for the block, packed for P.V, and the lane's sum
      float rs;
      u32x4 pf[4];
      auto expo = [&]() {
        const float nm = -m;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int kb = c >> 1, hh = c & 1;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p0 = fast_exp2(fmaf(s[kb][8 * hh + 2 * i], sc, nm));
            const float p1 = fast_exp2(fmaf(s[kb][8 * hh + 2 * i + 1], sc, nm));
            rs = c + i == 0 ? p0 : rs + p0;
            rs += p1;
            pf[c][i] = E::pack2(p0, p1);
          }
        }
      };
      // the block max is only formed when it can matter (see the head_dim-128
      // kernel): past the first key block, a lane sum of at most 2^kSlack
      // bounds every p by it, and m keeps
      bool full = jb == 0;
      if (!full) {
        expo();
        full = __any(!(rs <= kSumCap));
      }
      if (full) {
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
        mx = pair_max(mx);
        const float m_blk = mx * sc;
        if (__any(m_blk > m + kSlack)) {
          const float m_new = fmaxf(m, m_blk);
          const float alpha = fast_exp2(m - m_new);
          lsum *= alpha;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[nb][r] *= alpha;
          m = m_new;
        }
        expo();
      }
      lsum += rs;

      // O^T += V^T P^T, then the next block's S^T, at raised issue priority
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int st = 0; st < NPV; ++st) {
        const u32x4 A = st == 0 ? vp0 : st == 1 ? vp1 : v_operand(vt, st);
        o[st % NB] = E::mfma32(as_vec8<V8>(A), as_vec8<V8>(pf[st / NB]), o[st % NB]);
      }
      // the next block's first two K operands (its tile arrived during the
      // previous iteration; past the last block they are stale and dropped)
      const u32x4 kn0 = k_operand(kslot(jb + 1), 0), kn1 = k_operand(kslot(jb + 1), 1);
      // reads run two MFMAs ahead
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < NPV - 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      if (jb + 1 < nkw) qk_from(kslot(jb + 1), kn0, kn1);
      __builtin_amdgcn_s_setprio(0);
    }
    wait_vmem();
    __syncthreads();
  }

  // O = acc / l rounded to the input type (HTile:130-143), the correctly
  // rounded fp32 quotient by Markstein's correction, and the LSE
  const float ltot = pair_sum(lsum);
  if (row < a.Sq) {
    const float inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
    auto quot = [&](float x) {
      const float q0 = x * inv;
      return __builtin_fmaf(__builtin_fmaf(-q0, ltot, x), inv, q0);
    };
    uint16_t *op = (uint16_t *)a.o + b * a.os0 + h * a.os1 + row * a.os2;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const u32x2 pk = {E::pack2(quot(o[nb][4 * rq]), quot(o[nb][4 * rq + 1])),
                          E::pack2(quot(o[nb][4 * rq + 2]), quot(o[nb][4 * rq + 3]))};
        *(u32x2 *)(op + 32 * nb + 8 * rq + 4 * g) = pk;
      }
    if (g == 0 && a.lse)
      a.lse[((int64_t)b * a.Hq + h) * a.Sq + row] =
          ltot > 0.0f ? (m + log2f(ltot)) * kLn2 : -INFINITY;
  }
}

template <class E>
void launch_e(const AttnArgs &a, bool causal, hipStream_t s) {
  const dim3 grid((unsigned)(a.nqb * a.BH));
  if (causal)
    hipLaunchKernelGGL((attn_fwd_tile<E, 64, true>), grid, dim3(NT), 0, s, a);
  else
    hipLaunchKernelGGL((attn_fwd_tile<E, 64, false>), grid, dim3(NT), 0, s, a);
}

}  // namespace

hipError_t launch_attn_d64(const AttnArgs &a, int32_t dtype, bool causal, hipStream_t s) {
  if (dtype == 2)
    launch_e<Bf16Tag>(a, causal, s);
  else
    launch_e<F16Tag>(a, causal, s);
  return hipGetLastError();
}

}  // namespace neptune
