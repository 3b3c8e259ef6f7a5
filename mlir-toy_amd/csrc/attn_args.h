// attn_args.h — kernel-side argument block of the attention kernels
// (resolved by launch_attn_fwd from the validated AttnLaunch).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace neptune {

struct AttnArgs {
  const void *q, *k, *v;
  void *o;
  float *lse;
  int64_t qs0, qs1, qs2, ks0, ks1, ks2, vs0, vs1, vs2, os0, os1, os2;
  int32_t Hq, group, Sq, Sk, nqb, BH, off;  // off = Sk - Sq (causal diagonal)
  float scale2;                             // log2(e)/sqrt(D) unless given
};

// Launches the head_dim-128 16-bit kernel (attn_fwd_d128.hip); dtype 1 = f16,
// 2 = bf16; stages = LDS slots per operand (1, 2 or 3); kt = K stored
// [.., head_dim, seq] (ks2 is then the head_dim-row stride).
hipError_t launch_attn_d128(const AttnArgs &a, int32_t dtype, bool causal, int stages, bool kt,
                            hipStream_t s);

constexpr int kMaxAttnSplits = 32;  // a power of two (attn_combine)

// Short launches: the keys cut into splits whose states attn_combine merges,
// and (packed) the query heads of a KV head as one run of rows.
struct SplitArgs {
  int32_t nsplit;  // 0: the plain kernel; 1: no partials
  int32_t kbs;     // 64-key blocks per split
  int32_t packed;
  int32_t halves;  // 2: eight waves, four on each half of the split's keys
  float *po;       // [B * Hq * Sq, nsplit, head_dim]
  float *pml;      // [B * Hq * Sq, nsplit, 2]: (m, l)
};

// Launches the kernels of attn_fwd_tile.hip: head_dim 64, or (x.nsplit > 0)
// 64 or 128.
hipError_t launch_attn_tile(const AttnArgs &a, const SplitArgs &x, int32_t dtype, int head_dim,
                            bool causal, hipStream_t s);

}  // namespace neptune
