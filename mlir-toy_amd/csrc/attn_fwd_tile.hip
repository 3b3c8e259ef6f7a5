// attn_fwd_tile.hip — 16-bit HTile attention forward for gfx950: head_dim 64,
// and the cut form of short launches at head_dim 64 and 128.
//
// Semantics are those of attn_fwd.hip. The structure is that of the
// head_dim-128 kernel (attn_fwd_d128.hip): 256 threads = 4 waves, 128 query
// rows (32 per wave), 64-key blocks, K and V tiles HBM -> LDS by
// global_load_lds_dwordx4 into two slots per operand, the transposed products
//   S^T = K . Q^T   (A = K rows from LDS, B = Q^T in VGPRs)
//   O^T = V^T . P^T (A = V^T from LDS via ds_read_b64_tr_b16, B = P^T)
// on v_mfma_f32_32x32x16 (one query row per lane), and block j+1's QK^T in the
// MFMA stream of block j's P.V. At head_dim 128 the running max moves lazily,
// as in that kernel; at head_dim 64 it moves with every block that passes it,
// so that a row's largest p is 1 and takes no rounding to 16 bits.
//
// Bound: at head_dim 64 a key block's softmax (about 190 vector instructions a
// wave with the rescale of O) outweighs its 16 MFMAs (512 cycles). Two
// work-groups per CU (162-168 registers). Measured on the lazy form, three or
// four of them (127 registers, with the copies' rare tail computed in place)
// came within 3%, and a barrier for every second key block (four slots per
// operand) was 8% slower, so neither occupancy nor the barrier holds it back.
// Measured (GPU time, graph replays, against a kernel that staged K and V
// through registers and transposed V while writing it to LDS): B4 H16 S2048
// causal 64 -> 54.5 us (630 TFLOP/s), without the mask 105.6 -> 90.3 (760), B1
// H8 S4096 causal 83.5 -> 50.4, B4 H8 S55 5.35 -> 4.5. A lazy max here measured
// 51, 77.8, 41.2 and 4.3 us and 3-6% more error against 64 bits (f16, N(0, 1)),
// so it is not used.
#include "attn_args.h"
#include "attn_tile.h"
#include "kernels.h"

namespace neptune {
namespace {

// SPLIT: a work-group takes one split of the keys (x.kbs blocks) and, packed,
// rows that run through the heads of its KV head; with more than one split
// it leaves its unnormalised O and (m, l) for attn_combine. KW = 2: eight
// waves, four on each half of the keys, whose states merge in LDS lane to lane.
// 210 registers at head_dim 128 (two waves per SIMD). What it measured stands at
// attn_split, which chooses the cut.
template <class E, int HD, bool CAUSAL, bool SPLIT, int KW>
__global__ __launch_bounds__(NT * KW, 2 / KW) void attn_fwd_tile(AttnArgs a, SplitArgs x) {
  typedef typename E::vec8 V8;
  constexpr int TILE = TileLoader<HD>::TILE_BYTES;
  constexpr int ROWB = HD * 2;   // bytes per LDS row
  constexpr int NST = HD / 16;   // QK^T k-steps
  constexpr int NB = HD / 32;    // 32-wide head_dim blocks of O^T
  constexpr int NQK = 2 * NST, NPV = 4 * NB;  // MFMAs per key block
  // per key half: K slots 0 and 1, then V slots 0 and 1; block t uses slot t & 1
  __shared__ __attribute__((aligned(16))) uint8_t smem[KW * 4 * TILE];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = KW > 1 ? wave & 3 : wave, half = KW > 1 ? wave >> 2 : 0;
  const int lq = lane & 31, g = lane >> 5;
  const uint8_t *const kt0 = smem + half * 4 * TILE;
  const uint8_t *const vt0 = kt0 + 2 * TILE;
  auto kslot = [&](int t) { return kt0 + (t & 1) * TILE; };
  auto vslot = [&](int t) { return vt0 + (t & 1) * TILE; };

  // Work-group -> (kv head, split, query head of its group, query block): kv
  // heads fastest, so that (with a multiple of 8 of them) id % 8, the XCD,
  // fixes the kv head modulo 8 and all readers of a head's K and V share an
  // L2; the heaviest causal query blocks first
  const int BHk = a.BH / a.group;
  const int id = blockIdx.x;
  const int bhk = __builtin_amdgcn_readfirstlane(id % BHk);
  int rest = id / BHk, split = 0;
  if constexpr (SPLIT) {
    split = __builtin_amdgcn_readfirstlane(rest % x.nsplit);
    rest /= x.nsplit;
  }
  const bool packed = SPLIT && x.packed;
  const int heads = packed ? 1 : a.group;  // work-groups per row block and kv head
  const int qb = __builtin_amdgcn_readfirstlane(a.nqb - 1 - rest / heads);
  const int Hk = a.Hq / a.group;
  const int b = __builtin_amdgcn_readfirstlane(bhk / Hk);
  const int hk = bhk - b * Hk;
  const int h0 = __builtin_amdgcn_readfirstlane(hk * a.group + rest % heads);
  const uint16_t *kp = (const uint16_t *)a.k + b * a.ks0 + hk * a.ks1;
  const uint16_t *vp = (const uint16_t *)a.v + b * a.vs0 + hk * a.vs1;

  // this lane's row: query position pos of head h0 + hr (packed rows run
  // through the heads of the group, each all its positions)
  const int row = qb * BM + w * 32 + lq;
  const int rows = packed ? a.group * a.Sq : a.Sq;
  const int hr = packed ? row / a.Sq : 0, pos = row - hr * a.Sq;
  // the first and last position among rows r0 .. r0 + n - 1
  auto span = [&](int r0, int n, int *lo, int *hi) {
    const int r1 = min(r0 + n, rows) - 1;
    *lo = r0;
    *hi = r1;
    if (packed) {
      const int p0 = r0 / a.Sq, p1 = r1 / a.Sq;
      *lo = p0 == p1 ? r0 - p0 * a.Sq : 0;
      *hi = p0 == p1 ? r1 - p1 * a.Sq : a.Sq - 1;
    }
  };
  // key blocks kb0 .. kb0 + nv - 1 of the work-group, the first nkw of them
  // this wave's
  int kb0 = SPLIT ? split * x.kbs : 0;
  int nv = (a.Sk + BN - 1) / BN, nkw = nv, lo_w = 0;
  if (CAUSAL) {
    int lo, hi;
    span(qb * BM, BM, &lo, &hi);
    nv = min(nv, hi + a.off < 0 ? 0 : (hi + a.off) / BN + 1);
    span(qb * BM + w * 32, 32, &lo, &hi);
    nkw = min(nv, hi + a.off < 0 ? 0 : (hi + a.off) / BN + 1);
    lo_w = __builtin_amdgcn_readfirstlane(lo);
  }
  if (qb * BM + w * 32 >= rows) nkw = 0;
  if constexpr (SPLIT) {
    nv = min(max(nv - kb0, 0), x.kbs);
    nkw = min(max(nkw - kb0, 0), x.kbs);
  }
  // the trips of the key loop: with two halves, the first takes the odd block
  int trips = nv;
  if constexpr (KW > 1) {
    trips = (nv + 1) >> 1;
    const int first = half ? trips : 0, n = half ? nv - trips : trips;
    kb0 += first;
    nv = n;
    nkw = min(max(nkw - first, 0), n);
  }
  nv = __builtin_amdgcn_readfirstlane(nv);
  nkw = __builtin_amdgcn_readfirstlane(nkw);
  trips = KW > 1 ? __builtin_amdgcn_readfirstlane(trips) : nv;
  if constexpr (SPLIT) kb0 = __builtin_amdgcn_readfirstlane(kb0);

  const TileLoader<HD> kl = make_loader<HD, false>(kp, a.ks2, w, lane);
  const TileLoader<HD> vl = make_loader<HD, true>(vp, a.vs2, w, lane);
  auto load_k = [&](int t) { tile_to_lds<false>(kl, (kb0 + t) * BN, a.Sk, kslot(t), w); };
  auto load_v = [&](int t) { tile_to_lds<true>(vl, (kb0 + t) * BN, a.Sk, vslot(t), w); };
  if (nv > 0) load_k(0);
  if (nv > 1) load_k(1);
  if (nv > 0) load_v(0);

  // Q^T operand: k-step st covers head_dim 16 st + 8 g .. +7 of the row
  u32x4 qf[NST];
  {
    const uint16_t *qp = (const uint16_t *)a.q + b * a.qs0 + (h0 + hr) * a.qs1 + pos * a.qs2 + 8 * g;
#pragma unroll
    for (int st = 0; st < NST; ++st)
      qf[st] = row < rows ? *(const u32x4 *)(qp + 16 * st) : u32x4{0, 0, 0, 0};
  }

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

  for (int jb = 0; jb < trips; ++jb) {
    // K of block jb + 2 goes to the slot block jb's K has left, V of block
    // jb + 1 to the slot of block jb - 1's V
    if (jb + 2 < nv) load_k(jb + 2);
    if (jb + 1 < nv) load_v(jb + 1);
    if (jb < nkw) {
      // the first two V^T operands of this block's P.V, read before the softmax
      const uint8_t *vt = vslot(jb);
      const u32x4 vp0 = v_operand(vt, 0), vp1 = v_operand(vt, 1);
      const int key0 = (kb0 + jb) * BN;
      if ((key0 + BN > a.Sk) || (CAUSAL && key0 + BN - 1 > lo_w + a.off)) {
        // element (kb, r) holds key key0 + 4 g + c with c = 32 kb + 8 (r >> 2)
        // + (r & 3): it is masked when c passes the lane's last visible key
        int lim = a.Sk - 1 - key0 - 4 * g;
        if (CAUSAL) lim = min(lim, pos + a.off - key0 - 4 * g);
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
      auto raise_max = [&](float slack) {  // m to the block's max where that passes m + slack
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
        mx = pair_max(mx);
        const float m_blk = mx * sc;
        if (__any(m_blk > m + slack)) {
          const float m_new = fmaxf(m, m_blk);
          const float alpha = fast_exp2(m - m_new);
          lsum *= alpha;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[nb][r] *= alpha;
          m = m_new;
        }
      };
      if constexpr (HD == 64) {
        // the max of every block: a row's largest p is then exactly 1, with no
        // rounding to 16 bits
        raise_max(0.0f);
        expo();
      } else {
        // the block max is only formed when it can matter (see the head_dim-128
        // kernel): past the first key block, a lane sum of at most 2^kSlack
        // bounds every p by it, and m keeps
        bool full = jb == 0;
        if (!full) {
          expo();
          full = __any(!(rs <= kSumCap));
        }
        if (full) {
          raise_max(kSlack);
          expo();
        }
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

  float ltot = pair_sum(lsum);
  if constexpr (KW > 1) {
    // the second half's state to its row's wave of the first, lane to lane,
    // through the K/V slots (free since the loop's last barrier)
    f32x4 *const box = (f32x4 *)smem + (w * (4 * NB) * 64 + lane);
    f32x2 *const mlbox = (f32x2 *)(smem + KW * 4 * TILE) - 4 * 64 + (w * 64 + lane);
    if (half) {
#pragma unroll
      for (int v = 0; v < 4 * NB; ++v)
        box[v * 64] = f32x4{o[v >> 2][4 * (v & 3)], o[v >> 2][4 * (v & 3) + 1],
                            o[v >> 2][4 * (v & 3) + 2], o[v >> 2][4 * (v & 3) + 3]};
      *mlbox = f32x2{m, ltot};
    }
    __syncthreads();
    if (half) return;
    const f32x2 ml = *mlbox;
    const float M = fmaxf(m, ml[0]), w0 = fast_exp2(m - M), w1 = fast_exp2(ml[0] - M);
    ltot = ltot * w0 + ml[1] * w1;
    m = M;
#pragma unroll
    for (int v = 0; v < 4 * NB; ++v) {
      const f32x4 other = box[v * 64];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = 4 * (v & 3) + r;
        o[v >> 2][e] = fmaf(o[v >> 2][e], w0, other[r] * w1);
      }
    }
  }
  if (row < rows) {
    const int64_t grow = ((int64_t)b * a.Hq + h0 + hr) * a.Sq + pos;  // row of [B, Hq, Sq]
    if constexpr (SPLIT) {
      if (x.nsplit > 1) {  // this split's state, for attn_combine
        const int64_t part = grow * x.nsplit + split;
        if (trips > 0) {
          float *op = x.po + part * HD + 4 * g;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int rq = 0; rq < 4; ++rq)
              *(f32x4 *)(op + 32 * nb + 8 * rq) =
                  f32x4{o[nb][4 * rq], o[nb][4 * rq + 1], o[nb][4 * rq + 2], o[nb][4 * rq + 3]};
        }
        if (g == 0) *(f32x2 *)(x.pml + part * 2) = f32x2{m, ltot};
        return;
      }
    }
    // O = acc / l rounded to the input type (HTile:130-143), the correctly
    // rounded fp32 quotient by Markstein's correction, and the LSE
    const float inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
    auto quot = [&](float v) {
      const float q0 = v * inv;
      return __builtin_fmaf(__builtin_fmaf(-q0, ltot, v), inv, q0);
    };
    uint16_t *op = (uint16_t *)a.o + b * a.os0 + (h0 + hr) * a.os1 + pos * a.os2 + 4 * g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const u32x2 pk = {E::pack2(quot(o[nb][4 * rq]), quot(o[nb][4 * rq + 1])),
                          E::pack2(quot(o[nb][4 * rq + 2]), quot(o[nb][4 * rq + 3]))};
        *(u32x2 *)(op + 32 * nb + 8 * rq) = pk;
      }
    if (g == 0 && a.lse)
      a.lse[grow] = ltot > 0.0f ? (m + log2f(ltot)) * kLn2 : -INFINITY;
  }
}

// Combine of the splits' states: HD / 4 lanes per row, four head_dim elements
// each. M = max m_s, l = sum 2^(m_s - M) l_s, O = sum 2^(m_s - M) O_s / l; a
// split with l_s = 0 (no visible key) may have left no O_s and is passed over
// (weight -1); one whose weight is 0 by underflow is not, so that an infinity or
// NaN in its O_s reaches O as it does in an uncut launch. NS (a power of two) is
// at least the number of splits: every O_s is loaded before the first weight
// is known, so the row waits on memory once.
template <class E, int HD, int NS>
__global__ __launch_bounds__(NT) void attn_combine(AttnArgs a, SplitArgs x, int64_t nrows) {
  constexpr int LPR = HD / 4;
  const int64_t grow0 = (int64_t)blockIdx.x * (NT / LPR) + threadIdx.x / LPR;
  const int64_t grow = grow0 < nrows ? grow0 : nrows - 1;  // every lane takes part in the shuffles
  const int dl = threadIdx.x % LPR, d = 4 * dl;
  const f32x2 *ml = (const f32x2 *)x.pml + grow * x.nsplit;
  const float *po = x.po + grow * x.nsplit * HD + d;
  f32x4 os[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) os[s] = *(const f32x4 *)(po + (int64_t)min(s, x.nsplit - 1) * HD);
  // lane dl holds the state of splits dl, dl + LPR, ..
  constexpr int SPL = (NS + LPR - 1) / LPR;
  f32x2 st[SPL];
  float M = kNegFltMax;
#pragma unroll
  for (int i = 0; i < SPL; ++i) {
    const int s = dl + i * LPR;
    st[i] = s < x.nsplit ? ml[s] : f32x2{kNegFltMax, 0.0f};
    M = fmaxf(M, st[i][0]);
  }
#pragma unroll
  for (int off = LPR / 2; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, LPR));
  float l = 0.0f;
#pragma unroll
  for (int i = 0; i < SPL; ++i) {
    st[i][0] = st[i][1] == 0.0f ? -1.0f : fast_exp2(st[i][0] - M);  // the split's weight
    l = fmaf(st[i][0], st[i][1], l);
  }
#pragma unroll
  for (int off = LPR / 2; off >= 1; off >>= 1) l += __shfl_xor(l, off, LPR);
  f32x4 acc = {0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const float wgt = __shfl(st[s / LPR][0], s % LPR, LPR);
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = wgt < 0.0f ? acc[k] : fmaf(wgt, os[s][k], acc[k]);
  }
  if (grow0 >= nrows) return;
  const int64_t bh = grow / a.Sq;
  const int pos = (int)(grow - bh * a.Sq), b = (int)(bh / a.Hq), h = (int)(bh - (int64_t)b * a.Hq);
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  auto quot = [&](float v) {
    const float q0 = v * inv;
    return __builtin_fmaf(__builtin_fmaf(-q0, l, v), inv, q0);
  };
  uint16_t *op = (uint16_t *)a.o + b * a.os0 + h * a.os1 + pos * a.os2 + d;
  *(u32x2 *)op = u32x2{E::pack2(quot(acc[0]), quot(acc[1])), E::pack2(quot(acc[2]), quot(acc[3]))};
  if (d == 0 && a.lse) a.lse[grow] = l > 0.0f ? (M + log2f(l)) * kLn2 : -INFINITY;
}

template <class E, int HD, bool CAUSAL>
void launch_split(AttnArgs a, const SplitArgs &x, hipStream_t s) {
  const int BHk = a.BH / a.group;
  const int rows = x.packed ? a.group * a.Sq : a.Sq;
  a.nqb = (rows + BM - 1) / BM;
  const unsigned grid = (unsigned)a.nqb * (x.packed ? BHk : a.BH) * x.nsplit;
  if (x.halves > 1)
    hipLaunchKernelGGL((attn_fwd_tile<E, HD, CAUSAL, true, 2>), dim3(grid), dim3(2 * NT), 0, s, a,
                       x);
  else
    hipLaunchKernelGGL((attn_fwd_tile<E, HD, CAUSAL, true, 1>), dim3(grid), dim3(NT), 0, s, a, x);
  if (x.nsplit > 1) {
    const int64_t nrows = (int64_t)a.BH * a.Sq, per = NT / (HD / 4);
    auto k = x.nsplit <= 4    ? attn_combine<E, HD, 4>
             : x.nsplit <= 8  ? attn_combine<E, HD, 8>
             : x.nsplit <= 16 ? attn_combine<E, HD, 16>
                              : attn_combine<E, HD, kMaxAttnSplits>;
    hipLaunchKernelGGL(k, dim3((unsigned)((nrows + per - 1) / per)), dim3(NT), 0, s, a, x, nrows);
  }
}

template <class E>
void launch_e(const AttnArgs &a, const SplitArgs &x, int head_dim, bool causal, hipStream_t s) {
  if (x.nsplit > 0) {
    if (head_dim == 64)
      causal ? launch_split<E, 64, true>(a, x, s) : launch_split<E, 64, false>(a, x, s);
    else
      causal ? launch_split<E, 128, true>(a, x, s) : launch_split<E, 128, false>(a, x, s);
    return;
  }
  const dim3 grid((unsigned)(a.nqb * a.BH));
  if (causal)
    hipLaunchKernelGGL((attn_fwd_tile<E, 64, true, false, 1>), grid, dim3(NT), 0, s, a, x);
  else
    hipLaunchKernelGGL((attn_fwd_tile<E, 64, false, false, 1>), grid, dim3(NT), 0, s, a, x);
}

}  // namespace

hipError_t launch_attn_tile(const AttnArgs &a, const SplitArgs &x, int32_t dtype, int head_dim,
                            bool causal, hipStream_t s) {
  if (dtype == 2)
    launch_e<Bf16Tag>(a, x, head_dim, causal, s);
  else
    launch_e<F16Tag>(a, x, head_dim, causal, s);
  return hipGetLastError();
}

}  // namespace neptune
