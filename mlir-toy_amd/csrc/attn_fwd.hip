// attn_fwd.hip — the HTile flash-attention tile program on gfx950.
//
// Semantics: tests/data/flash_attention_htile.mlir:26-143 (one program per
// (128-row query block, head, batch); K/V streamed in 64-key blocks; fp32
// online softmax in the exp2 domain; P rounded to the 16-bit input type
// before P.V; O = acc / l rounded on store). Additions the reference lacks:
// causal masking (bottom-right aligned), per-row logsumexp, grouped KV heads,
// strided tensors and ragged sequence lengths.
//
// This file holds the fp32 kernel and the choice of kernel; the 16-bit ones
// are attn_fwd_d128.hip (head_dim 128) and attn_fwd_tile.hip (head_dim 64).
#include <algorithm>

#include "device_common.h"
#include "kernels.h"
#include "attn_args.h"

namespace neptune {
namespace {

// fp32 path (any F32 request). v_mfma_f32_16x16x4_f32 forms both products
// in fp32 (fp32 operands, products and sums: the HTile recurrence with no
// rounding of P, the input type being fp32).
//
// A work-group takes 16 * NQ query rows, and its NW waves share out the keys:
// wave w runs the online softmax (m, l, O) over the 16-key blocks w, w + NW,
// .. for all of those rows, and the NW states of a row are merged at the end
// through LDS in the exp2 domain (M = max m_w, l = sum 2^(m_w - M) l_w, the
// same for O). As in the 16-bit kernels each wave forms the transposed products
//   S^T = K . Q^T    O^T = V^T . P^T
// so lane (i = lane % 16, g = lane / 16) holds query i's scores of keys 4 g + r
// (r = 0..3) of the block, which is the B operand of P.V as it stands. No key
// or value is read by two waves, so K and V go straight from memory to the A
// operand registers, 16 bytes a lane: the k index of a product may be any
// order that both operands share, and a row index any order the result is
// read back in, so a lane takes four neighbouring head_dim elements of its
// key (K), and four neighbouring head_dim rows of V^T. K of the next block is
// loaded while this one's softmax and P.V run, V at the top of its own block.
//
// Bound: fp32 MFMA, D/2 instructions of 32 cycles per 16 keys and 16 rows;
// they run on the vector ALU's own multipliers, so the softmax does not hide
// behind them. The NQ column blocks share every K and V load. Measured (GPU
// time, against a vector-ALU kernel that held one key's whole dot product
// in a lane): B2 H12 S1500 D64 causal 361 -> 81 us (85 TFLOP/s; a large fp32
// GEMM reaches 154 on this card), B2 H16 S1024 D128 1434 -> 162 us (106
// TFLOP/s), B1 H1 S128 D64 10.3 -> 4.9 us (three quarters of it launch
// latency). Reading K and V by ranges (f32_rows) took the 64-bit address of
// every row, 15 quarter-rate multiplies per 16 keys, out of the loop: the first
// two 81 -> 78 and 164 -> 148 us, B4 H16 S800 D32 61.7 -> 55.3, one query over
// 2048 keys of 8 heads, D128, 49.3 -> 39.4.
constexpr int F32_KB = 16;  // keys per block and wave
// A wave adds up P.V over F32_STRETCH blocks, then adds that to the sum of its
// earlier stretches, kept in LDS: the rounding of a sum of n terms grows with
// sqrt(n), and 96 terms at a time keep it below that of the vector-ALU kernel,
// which summed Sk / 16 terms in each of 16 lanes. Relative error against 64
// bits (1e-7; N(0, 1), no mask; that kernel / one sum per wave / stretches): S
// 2048 D32 3.25 / 4.47 / 2.56, D64 3.75 / 4.58 / 2.76, D128 4.62 / 4.81 / 3.15; S
// 512 D32 2.52 / 2.59 / 2.29. The stretches cost up to 4% of the time (B2 H12
// S1500 D64 causal 75.0 -> 78.1 us, the figures above being without them; D128
// no mask and D32 1%); four blocks instead of six cost 1% more.
constexpr int F32_STRETCH = 6;
// The split of the work by the number of 32-row blocks of the launch. Below
// the line the GPU is short of work-groups and a wave's serial key loop sets
// the time, so 16-row work-groups cut the keys eight ways; above it the
// matrix units are full and 32-row work-groups of 4 waves read K and V half
// as often. Measured (us, 16-row / 32-row; D = 64, then 32 and 128): no mask 128
// blocks (8 heads, S 512) 9.8 / 14.0, 6.5 / 8.8, 16.6 / 23.6; 256 (16 heads)
// 16.6 / 14.9, 10.2 / 9.5, 30.6 / 24.3; causal, where the late blocks hold most of
// the work, 256 13.5 / 14.5, 8.5 / 9.1, 23.0 / 24.2; 512 (32 heads) 22.4 / 19.2,
// 13.7 / 11.9, 42.9 / 33.5; 512 (16 heads, S 1024) 32.3 / 31.0, 20.5 / 18.8, 62.4
// / 56.0.
constexpr int64_t F32_FILL = 256, F32_FILL_CAUSAL = 512;

template <int N>
struct F32Vec;
template <>
struct F32Vec<4> { typedef f32x4 type; };
template <>
struct F32Vec<2> { typedef f32x2 type; };

// N consecutive floats; VEC: the address is a multiple of 4 N bytes
template <int N, bool VEC>
__device__ inline typename F32Vec<N>::type load_f32(const float *p) {
  typedef typename F32Vec<N>::type V;
  if constexpr (VEC) return *(const V *)p;
  V v;
#pragma unroll
  for (int e = 0; e < N; ++e) v[e] = p[e];
  return v;
}

// The rows row0 .. row0 + F32_KB - 1 of one head's K or V (seq rows, stride
// floats apart), to the end of the last one that exists: rows beyond it start at
// or past the range's end (stride >= D), where loads return 0.
__device__ inline __amdgpu_buffer_rsrc_t f32_rows(const float *head, int64_t stride, int row0,
                                                  int seq, int D) {
  const int n = max(min(seq - row0, F32_KB), 0);
  const int bytes = max(4 * ((n - 1) * (int)stride + D), 0);  // n = 0: stride >= D
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(head + row0 * stride), (short)0,
                                           bytes, 0x00020000);
}

// VEC: 16-byte loads and stores (every base and stride a multiple of 16
// bytes, and K and V rows as f32_rows addresses them); otherwise one element
// each. At head_dim 32 the causal form is held to five waves per SIMD (left to
// itself it takes 98 registers, two too many: B4 H16 S800 33.3 / 30.3 us)
template <int D, bool CAUSAL, int NQ, int NW, bool VEC>
__global__ __launch_bounds__(64 * NW, D == 32 && CAUSAL && NQ == 2 ? 5 : 1) void attn_fwd_f32(
    AttnArgs a) {
  constexpr int NM = D / 16;             // 16-wide head_dim blocks
  constexpr int VW = NM < 4 ? NM : 4;    // head_dim elements per V load
  constexpr int VL = NM / VW;            // V loads per key
  constexpr int ROWS = 16 * NQ;
  constexpr int OP = D + 4;              // row pitch of the merge buffer
  typedef typename F32Vec<VW>::type VV;
  __shared__ __attribute__((aligned(16))) float mo[NW][ROWS][OP];
  __shared__ float mm[NW][ROWS], ml[NW][ROWS];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int id = blockIdx.x;
  // heaviest causal query blocks first
  const int qb = CAUSAL ? a.nqb - 1 - id / a.BH : id / a.BH;
  const int bh = id % a.BH;
  const int b = bh / a.Hq, h = bh % a.Hq, hk = h / a.group;
  const float *qp = (const float *)a.q + b * a.qs0 + h * a.qs1;
  const float *kp = (const float *)a.k + b * a.ks0 + hk * a.ks1;
  const float *vp = (const float *)a.v + b * a.vs0 + hk * a.vs1;
  const int row0 = qb * ROWS;

  int nkb = (a.Sk + F32_KB - 1) / F32_KB;
  if (CAUSAL) {
    const int last = min(row0 + ROWS, a.Sq) - 1 + a.off;
    nkb = min(nkb, last < 0 ? 0 : last / F32_KB + 1);
  }

  // VEC: a block's rows are read through a buffer resource that begins with the
  // block and ends with its last row that exists (f32_rows), so a lane's offsets
  // are fixed and rows past the end read 0. Otherwise rows past the end read the
  // tensor's last one. Either way no load is guarded, and such keys are masked.
  const int krow = i * (int)a.ks2 + 4 * g, vcol = VW * i, vrow = (int)a.vs2;
  f32x4 kf[NM];
  auto load_k = [&](int kb) {
    if constexpr (VEC) {
      const auto r = f32_rows(kp, a.ks2, kb * F32_KB, a.Sk, D);
#pragma unroll
      for (int m = 0; m < NM; ++m)
        kf[m] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, 4 * krow + 64 * m, 0, 0));
    } else {
      const float *r = kp + min(kb * F32_KB + i, a.Sk - 1) * a.ks2 + 4 * g;
#pragma unroll
      for (int m = 0; m < NM; ++m) kf[m] = load_f32<4, VEC>(r + 16 * m);
    }
  };
  load_k(w);
  f32x4 qf[NQ][NM];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const float *r = qp + min(row0 + 16 * n + i, a.Sq - 1) * a.qs2 + 4 * g;
#pragma unroll
    for (int m = 0; m < NM; ++m) qf[n][m] = load_f32<4, VEC>(r + 16 * m);
  }

  // O^T block c of query block n: element r is head_dim row 4 g + r of the
  // block, which is head_dim VW (4 g + r) + c % VW + 64 (c / VW)
  f32x4 o[NQ][NM];
  float m[NQ], l[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    m[n] = kNegFltMax;
    l[n] = 0.0f;
#pragma unroll
    for (int c = 0; c < NM; ++c) o[n][c] = f32x4{0, 0, 0, 0};
  }
  const float sc = a.scale2;

  // the sums of the earlier stretches, in this wave's part of mo (value v of the
  // lane at 64 v), scaled by the max of their last block (in its part of mm)
  int since = 0;  // blocks since the last stretch ended
  bool banked = false;
  auto bank = [&](int v) { return (f32x4 *)&mo[w][0][0] + 64 * v + lane; };
  auto add_bank = [&](int n) {
    const float keep = fast_exp2(mm[w][16 * n + i] - m[n]);
#pragma unroll
    for (int c = 0; c < NM; ++c) {
      const f32x4 old = *bank(n * NM + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[n][c][r] = fmaf(old[r], keep, o[n][c][r]);
    }
  };

  for (int kb = w; kb < nkb; kb += NW) {
    const int key0 = kb * F32_KB;
    VV vf[4][VL];  // V of keys 4 g + r
    if constexpr (VEC) {
      const auto rows = f32_rows(vp, a.vs2, key0, a.Sk, D);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < VL; ++c) {
          const int at = 4 * ((4 * g + r) * vrow + vcol) + 256 * c;
          if constexpr (VW == 4)
            vf[r][c] = __builtin_bit_cast(VV, __builtin_amdgcn_raw_buffer_load_b128(rows, at, 0, 0));
          else
            vf[r][c] = __builtin_bit_cast(VV, __builtin_amdgcn_raw_buffer_load_b64(rows, at, 0, 0));
        }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float *vr = vp + min(key0 + 4 * g + r, a.Sk - 1) * a.vs2 + VW * i;
#pragma unroll
        for (int c = 0; c < VL; ++c) vf[r][c] = load_f32<VW, VEC>(vr + 64 * c);
      }
    }
    // two chains of D / 2 terms per score: half the rounding of one chain of D,
    // and no product waits for the one just before it
    f32x4 s[NQ], s2[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) s[n] = s2[n] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < NM; c += 2)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
          s[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][e], qf[n][c][e], s[n], 0, 0, 0);
          s2[n] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c + 1][e], qf[n][c + 1][e], s2[n], 0, 0, 0);
        }
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[n][r] += s2[n][r];
    // unconditionally (past the last block the rows are zeros, or the tensor's
    // last one again): a branch would make the compiler wait for these loads
    // before P.V
    load_k(kb + NW);
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      if (key0 + F32_KB > a.Sk || (CAUSAL && key0 + F32_KB - 1 > row0 + 16 * n + a.off)) {
        int lim = a.Sk - 1 - key0 - 4 * g;  // the lane's last visible r
        if (CAUSAL) lim = min(lim, row0 + 16 * n + i + a.off - key0 - 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r > lim) s[n][r] = -INFINITY;
      }
      // the running max moves only when a block's max passes it by more than
      // 8 (log2 units): in between p <= 2^8, which fp32 holds as well. Past
      // the first block it is formed only when a lane's sum says it may.
      float rs = 0.0f;
      f32x4 p;
      auto expo = [&]() {
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = fast_exp2(fmaf(s[n][r], sc, -m[n]));
        rs = (p[0] + p[1]) + (p[2] + p[3]);
      };
      bool full = kb == w;
      if (!full) {
        expo();
        full = __any(!(rs <= 256.0f));
      }
      if (full) {
        const float mx = max_xor32(
            max_xor16(fmaxf(fmaxf(s[n][0], s[n][1]), fmaxf(s[n][2], s[n][3]))));
        const float m_blk = mx * sc;
        if (__any(m_blk > m[n] + 8.0f)) {
          const float m_new = fmaxf(m[n], m_blk);
          const float alpha = fast_exp2(m[n] - m_new);
          l[n] *= alpha;
#pragma unroll
          for (int c = 0; c < NM; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[n][c][r] *= alpha;
          m[n] = m_new;
        }
        expo();
      }
      l[n] += rs;
      s[n] = p;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < NM; ++c)
#pragma unroll
        for (int n = 0; n < NQ; ++n)
          o[n][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r][c / VW][c % VW], s[n][r], o[n][c],
                                                         0, 0, 0);
    if (++since == F32_STRETCH) {
      since = 0;
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        if (banked) add_bank(n);
        mm[w][16 * n + i] = m[n];
#pragma unroll
        for (int c = 0; c < NM; ++c) {
          *bank(n * NM + c) = o[n][c];
          o[n][c] = f32x4{0, 0, 0, 0};
        }
      }
      banked = true;
    }
  }
  if (banked)
#pragma unroll
    for (int n = 0; n < NQ; ++n) add_bank(n);

  // merge the waves' states
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    l[n] += __shfl_xor(l[n], 16, 64);
    l[n] += __shfl_xor(l[n], 32, 64);
    if (g == 0) {
      mm[w][16 * n + i] = m[n];
      ml[w][16 * n + i] = l[n];
    }
  }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    float M = kNegFltMax;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, mm[ww][16 * n + i]);
    const float wgt = fast_exp2(m[n] - M);  // a wave with no visible key: l = 0, O = 0
#pragma unroll
    for (int c = 0; c < VL; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        VV v;
#pragma unroll
        for (int e = 0; e < VW; ++e) v[e] = o[n][c * VW + e][r] * wgt;
        *(VV *)&mo[w][16 * n + i][64 * c + VW * (4 * g + r)] = v;
      }
  }
  __syncthreads();
  constexpr int CPR = D / 4;  // 16-byte chunks per row
  for (int e = tid; e < ROWS * CPR; e += 64 * NW) {
    const int rl = e / CPR, d = 4 * (e % CPR), row = row0 + rl;
    if (row >= a.Sq) break;  // e, and with it the row, only grows
    float M = kNegFltMax;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, mm[ww][rl]);
    float ltot = 0.0f;
    f32x4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      ltot = fmaf(fast_exp2(mm[ww][rl] - M), ml[ww][rl], ltot);
      const f32x4 v = *(const f32x4 *)&mo[ww][rl][d];
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] += v[k];
    }
    // the correctly rounded quotient acc / l (HTile:130-143): q = acc * (1/l)
    // with the correctly rounded reciprocal, then one residual step
    // q + fma(-q, l, acc) * (1/l) (Markstein's correction)
    const float inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
    float *op = (float *)a.o + b * a.os0 + h * a.os1 + row * a.os2 + d;
    f32x4 res;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float q0 = acc[k] * inv;
      res[k] = __builtin_fmaf(__builtin_fmaf(-q0, ltot, acc[k]), inv, q0);
    }
    if constexpr (VEC) {
      *(f32x4 *)op = res;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) op[k] = res[k];
    }
    if (a.lse && d == 0)
      a.lse[((int64_t)b * a.Hq + h) * a.Sq + row] = ltot > 0.0f ? row_lse(M, ltot) : -INFINITY;
  }
}

template <int D, bool CAUSAL>
void launch_f32_d(AttnArgs args, bool vec, hipStream_t s) {
  auto go = [&](auto NQ, auto NW) {
    constexpr int nq = decltype(NQ)::value, nw = decltype(NW)::value;
    args.nqb = (args.Sq + 16 * nq - 1) / (16 * nq);
    auto k = vec ? attn_fwd_f32<D, CAUSAL, nq, nw, true> : attn_fwd_f32<D, CAUSAL, nq, nw, false>;
    hipLaunchKernelGGL(k, dim3((unsigned)(args.nqb * args.BH)), dim3(64 * nw), 0, s, args);
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  using I8 = std::integral_constant<int, 8>;
  const int64_t groups = (int64_t)((args.Sq + 31) / 32) * args.BH;
  if (groups >= (CAUSAL ? F32_FILL_CAUSAL : F32_FILL))
    go(I2{}, I4{});
  else
    go(I1{}, I8{});
}

template <int D>
void launch_f32(const AttnArgs &args, bool causal, bool vec, hipStream_t s) {
  if (causal)
    launch_f32_d<D, true>(args, vec, s);
  else
    launch_f32_d<D, false>(args, vec, s);
}

}  // namespace

bool attn_supported(const AttnLaunch &a, const char **why) {
  if (a.dtype == 0) {  // F32
    if (a.head_dim != 32 && a.head_dim != 64 && a.head_dim != 128) {
      *why = "fp32 attention supports head_dim 32, 64 or 128";
      return false;
    }
  } else if (a.head_dim != 64 && a.head_dim != 128) {
    *why = "16-bit attention supports head_dim 64 or 128";
    return false;
  }
  const bool d128 = a.dtype != 0 && a.head_dim == 128;
  if (a.stages != 2 && !d128) {
    *why = "pipeline_stages other than 2 applies to the head_dim-128 16-bit kernel";
    return false;
  }
  if (a.k_dim_order != 0) {
    if (!d128) {
      *why = "k_dim_order 1 applies to the head_dim-128 16-bit kernel";
      return false;
    }
    if (a.seq_kv % 8) {
      *why = "k_dim_order 1 needs seq_kv to be a multiple of 8";
      return false;
    }
  }
  if (a.seq_q > (int64_t)1 << 30 || a.seq_kv > (int64_t)1 << 30 ||
      a.batch * a.heads_q > (int64_t)1 << 24) {
    *why = "sequence or batch*heads too large for one launch";
    return false;
  }
  // The head_dim-128 kernel addresses a full K or V tile from a per-block
  // base plus per-lane 32-bit byte offsets: up to row 63 of a 64-key tile
  // (row 127 of a 128-row head_dim-major K tile) and 256 bytes into it.
  if (d128) {
    const int64_t klast = a.k_dim_order ? 127 : 63;
    if (klast * a.ks[2] * 2 + 256 > (int64_t)0xffffffff || 63 * a.vs[2] * 2 + 256 > (int64_t)0xffffffff) {
      *why = "K or V row stride too large: a 64-key tile must span less than 4 GiB";
      return false;
    }
  }
  // a dispatch covers at most 2^32 - 1 work-items: one 256-thread work-group
  // per 128 query rows and (batch, head) (the most any 16-bit path launches),
  // one 256-thread work-group per 16 rows for fp32 (twice what the 32-row form
  // launches; the 16-row form, 512 threads per 16 rows, is kept to fewer than
  // F32_FILL_CAUSAL 32-row blocks, 2^19 work-items)
  const int64_t rows = a.dtype == 0 ? 16 : 128;
  if ((a.seq_q + rows - 1) / rows * (a.batch * a.heads_q) * 256 > (int64_t)0xffffffff) {
    *why = "batch*heads*seq_q too large for one launch";
    return false;
  }
  return true;
}

// The cut of a 16-bit launch that leaves the GPU short of work-groups (at 128
// query rows each), by sizes alone:
//
// - Packing: the heads of a KV head share its K and V, so their rows may run
//   on into one another's 128-row blocks. It is used when that takes fewer
//   blocks, except under the causal mask over a long run of queries, where a
//   block across two heads would see the keys of the later head's last rows.
// - Splits: a work-group's time is its chain of 64-key blocks, so with at most
//   one work-group per CU the chain is cut. The count is the one with the
//   least estimated time: a key block takes 1.05 us alone on a CU and 1.65 us
//   beside another work-group (head_dim 64: 0.94 and 1.35), a launch 3 us, the
//   combine 4.5 us, and the states move at 5 TB/s. Measured alone 1.04 (0.95),
//   beside another 1.65 to 2.0 (1.35 to 1.5) with K and V from memory. A cut has
//   to promise 5%. Measured (us, one piece / chosen cut / its count): 1 x 32/8
//   heads, 250 queries over 8000 keys 135 / 47.2 / 8; 500 over 4000 71 / 46 / 4;
//   1 x 8 heads, 128 over 12000 197 / 23.3 / 27; 8 x 32/4 heads, 1 over 4000 68 /
//   17.7 / 16; head_dim 64, 1 x 16/4, 250 over 8000 126 / 27.8 / 16; 1 x 4, 2048
//   over 2048 causal 35.9 / 18.9 / 8; 3 x 4, 2 over 430 9.6 / 6.9 / 7. Where it
//   stays whole: 1 x 32 heads, 1000 over 1000 causal 23.0 / 31.7 with two splits;
//   1 x 32/8, 256 over 512 14.6 / 17.9 (head_dim 64: 18.5 / 25.5, 11.3 / 13.1).
// - Halves: a launch of at most one work-group per CU that stays whole has
//   eight waves per work-group, four on each half of the keys, merged in LDS.
//   The waves of a SIMD run in step, so their matrix and vector work overlaps
//   less than two work-groups' (1.75 us a block pair, 1.3 at head_dim 64, and
//   1.5 us for the merge; under splits it lost to more of them: 500 over 4000
//   58.1 / 46). Measured (us, four waves / eight): 1 x 16 heads causal S 1500
//   31.1 / 27.3, S 2000 39.1 / 33.8, 1 x 32 S 1000 23.5 / 22.1, S 640 17.1 /
//   16.9, S 512 14.9 / 15.3 (too few blocks: four); head_dim 64 S 1500 28.1 /
//   22.9, S 2000 35.9 / 28.6, 1 x 32 S 1000 21.0 / 18.0, S 640 14.9 / 13.3, S 512
//   12.7 / 11.8.
// - Without the mask the head_dim-128 kernel runs two query blocks per
//   work-group; up to 512 blocks they are better apart (1 x 4 heads, 512
//   over 512: 25.3 / 13.8).
AttnSplit attn_split(const AttnLaunch &L, bool partials) {
  AttnSplit p;
  if (L.dtype == 0 || L.k_dim_order != 0) return p;
  const bool causal = L.causal != 0, d128 = L.head_dim == 128;
  const int64_t group = L.heads_q / L.heads_kv, BHk = L.batch * L.heads_kv;
  const int64_t rows = L.batch * L.heads_q * L.seq_q;
  const int64_t plain = (L.seq_q + 127) / 128 * group * BHk;
  const int64_t packed = (L.seq_q * group + 127) / 128 * BHk;
  const int64_t nkb = (L.seq_kv + 63) / 64;
  constexpr int64_t kSlots = 512;  // two work-groups on each of 256 CUs
  p.packed = packed < plain && (!causal || L.seq_q < 128 || 4 * L.seq_q <= L.seq_kv);
  const int64_t wgs = p.packed ? packed : plain;
  // estimated nanoseconds with the keys cut into ns splits
  auto cost = [&](int64_t ns) {
    const int64_t step = wgs * ns <= kSlots / 2 ? (d128 ? 1050 : 940) : (d128 ? 1650 : 1350);
    int64_t t = (nkb + ns - 1) / ns * step;
    if (ns > 1) {
      // states written and read: causal blocks leave the splits past them empty
      const int64_t empty = causal ? (ns - 1) * std::min(L.seq_q, L.seq_kv) : 0;
      t += 3000 + 4500 +
           (int64_t)((double)rows * (L.head_dim + 2) * 8 / 5000 *
                     (ns - (double)empty / (2.0 * L.seq_kv)));
    } else {
      t += 3000;
    }
    return t;
  };
  int64_t best = 1;
  if (wgs <= kSlots / 2) {
    if (nkb >= (d128 ? 10 : 8)) p.halves = 2;
    const int64_t one =
        p.halves == 2 ? std::min(cost(1), 4500 + (nkb + 1) / 2 * (d128 ? 1750 : 1300)) : cost(1);
    int64_t best_t = one * 95 / 100;
    for (int64_t ns = 2;
         partials && ns <= kMaxAttnSplits && wgs * ns <= kSlots && ns <= nkb; ++ns)
      if (cost(ns) < best_t) {
        best_t = cost(ns);
        best = ns;
        p.halves = 1;
      }
  }
  if (best == 1 && p.halves == 1 && !(p.packed && 2 * packed <= plain) &&
      !(d128 && !causal && wgs <= kSlots))
    return AttnSplit();
  p.kbs = (int32_t)((nkb + best - 1) / best);
  p.nsplit = (int32_t)((nkb + p.kbs - 1) / p.kbs);
  if (p.nsplit > 1) p.bytes = (size_t)rows * p.nsplit * (L.head_dim + 2) * 4;
  return p;
}

hipError_t launch_attn_fwd(const AttnLaunch &L, const AttnSplit &split, void *workspace,
                           hipStream_t s) {
  AttnArgs a;
  a.q = L.q;
  a.k = L.k;
  a.v = L.v;
  a.o = L.o;
  a.lse = L.lse;
  a.qs0 = L.qs[0]; a.qs1 = L.qs[1]; a.qs2 = L.qs[2];
  a.ks0 = L.ks[0]; a.ks1 = L.ks[1]; a.ks2 = L.ks[2];
  a.vs0 = L.vs[0]; a.vs1 = L.vs[1]; a.vs2 = L.vs[2];
  a.os0 = L.os[0]; a.os1 = L.os[1]; a.os2 = L.os[2];
  a.Hq = (int32_t)L.heads_q;
  a.group = (int32_t)(L.heads_q / L.heads_kv);
  a.Sq = (int32_t)L.seq_q;
  a.Sk = (int32_t)L.seq_kv;
  a.BH = (int32_t)(L.batch * L.heads_q);
  a.off = (int32_t)(L.seq_kv - L.seq_q);
  a.scale2 = L.scale_log2;
  const bool causal = L.causal != 0;
  if (L.dtype == 0) {
    bool vec = true;
    for (int i = 0; i < 3; ++i)
      vec = vec && L.qs[i] % 4 == 0 && L.ks[i] % 4 == 0 && L.vs[i] % 4 == 0 && L.os[i] % 4 == 0;
    // f32_rows: rows that do not overlap (one past the end would start inside
    // the range), a block's offsets in 31 bits
    for (int64_t st : {L.ks[2], L.vs[2]}) vec = vec && st >= L.head_dim && st < (1 << 25);
    for (const void *p : {L.q, L.k, L.v, (const void *)L.o}) vec = vec && ((uintptr_t)p & 15u) == 0;
    switch (L.head_dim) {
      case 32: launch_f32<32>(a, causal, vec, s); break;
      case 64: launch_f32<64>(a, causal, vec, s); break;
      default: launch_f32<128>(a, causal, vec, s); break;
    }
  } else {
    a.nqb = (int32_t)((L.seq_q + 127) / 128);  // blocks of 128 query rows
    if (split.nsplit > 0 || L.head_dim == 64) {
      SplitArgs x;
      x.nsplit = split.nsplit;
      x.kbs = split.kbs;
      x.packed = split.packed;
      x.halves = split.halves;
      x.po = (float *)workspace;
      x.pml = x.po + (size_t)(L.batch * L.heads_q * L.seq_q) * split.nsplit * L.head_dim;
      return launch_attn_tile(a, x, L.dtype, (int)L.head_dim, causal, s);
    }
    return launch_attn_d128(a, L.dtype, causal, L.stages, L.k_dim_order != 0, s);
  }
  return hipGetLastError();
}

}  // namespace neptune
