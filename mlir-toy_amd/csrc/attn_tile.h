// attn_tile.h — what the tiled 16-bit attention kernels share: the block
// shape, the K/V tile copies into LDS and the in-wave row reductions.
#pragma once

#include "device_common.h"
#include "lds_dma.h"

namespace neptune {
namespace {

constexpr int BM = 128;            // query rows per work-group (HTile %c128), 32 per wave
constexpr int BN = 64;             // keys per block (HTile %c64)
constexpr int NT = 256;            // threads per work-group
constexpr float kSlack = 8.0f;     // lazy-rescale threshold (log2 units)
constexpr float kSumCap = 256.0f;  // 2^kSlack: a lane's block sum at most this skips the max

// LDS tiles (K stored [.., seq, head_dim], and V) are 64 rows of HD 16-bit
// elements in 16-byte units, XOR-swizzled per row so that the DMA writes (one
// 1 KiB chunk, whole rows) and the MFMA operand reads are bank-conflict free.
// 256 bytes hold one row (head_dim 128) or two (64): the swizzle spreads the
// 16 rows that read one unit together (K), and the four rows whose 64-byte
// runs are transposed together (V), over them.
template <int HD, bool IS_V>
__device__ inline int tile_swizzle(int r) {
  if constexpr (HD == 128)
    return IS_V ? (r & 3) << 2 : r & 15;
  else
    return IS_V ? ((r >> 1) & 1) << 2 : (r >> 1) & 7;
}

// Wave w copies rows [16w, 16w+16) of a tile straight into LDS, in 1 KiB
// chunks. Full blocks take a wave-uniform base pointer plus per-lane 32-bit
// offsets fixed for the whole kernel, so issuing a chunk costs no vector ALU
// work; a block that runs past the end of the sequence re-reads the last row
// instead (its scores are masked, so its P is exactly 0).
template <int HD>
struct TileLoader {
  static constexpr int UNITS = HD / 8;            // 16-byte units per row
  static constexpr int RPC = 64 / UNITS;          // rows per chunk
  static constexpr int CHUNKS = 16 / RPC;         // chunks per wave and tile
  static constexpr int TILE_BYTES = BN * HD * 2;
  const char *base;      // element (0, 0) of this (batch, head)
  int64_t row_bytes;     // key stride in bytes
  uint32_t off[CHUNKS];  // per-lane byte offset of chunk c within a full block
  bool wide;             // a tile spans 4 GiB or more: off[] does not hold its offsets
  int lane_row;          // row of chunk 0 for this lane
  int unit;              // unit within the row this lane fills
};

template <int HD, bool IS_V>
__device__ inline TileLoader<HD> make_loader(const uint16_t *src, int64_t stride, int w, int lane) {
  typedef TileLoader<HD> T;
  T t;
  t.base = (const char *)src;
  t.row_bytes = stride * 2;
  // head_dim 128 is refused at such strides
  t.wide = HD == 64 && (BN - 1) * t.row_bytes + HD * 2 > (int64_t)0xffffffff;
  t.lane_row = 16 * w + lane / T::UNITS;
  t.unit = lane & (T::UNITS - 1);
#pragma unroll
  for (int c = 0; c < T::CHUNKS; ++c) {
    const int r = t.lane_row + T::RPC * c;
    const int unit = t.unit ^ tile_swizzle<HD, IS_V>(r);
    t.off[c] = (uint32_t)((int64_t)r * t.row_bytes + unit * 16);
  }
  return t;
}

template <bool IS_V, int HD>
__device__ inline void tile_to_lds(const TileLoader<HD> &t, int key0, int Sk, const uint8_t *tile,
                                   int w) {
  typedef TileLoader<HD> T;
  if (key0 + BN <= Sk && !t.wide) {
    const char *blk = t.base + (int64_t)key0 * t.row_bytes;
#pragma unroll
    for (int c = 0; c < T::CHUNKS; ++c)
      dma16_sbase(blk, t.off[c], lds_offset(tile + (T::CHUNKS * w + c) * 1024));
  } else {
#pragma unroll
    for (int c = 0; c < T::CHUNKS; ++c) {
      const int r = t.lane_row + T::RPC * c;
      const int unit = t.unit ^ tile_swizzle<HD, IS_V>(r);
      const int key = min(key0 + r, Sk - 1);
      dma16(t.base + (int64_t)key * t.row_bytes + unit * 16,
            lds_offset(tile + (T::CHUNKS * w + c) * 1024));
    }
  }
}

__device__ inline void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)

// (lane, lane ^ 32) pair reductions through v_permlane32_swap
__device__ inline float pair_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float pair_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace
}  // namespace neptune
