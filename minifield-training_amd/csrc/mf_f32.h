// Shared pieces of the fp32 attention kernels: the work unit (32 rows of one
// head), operand tiles in LDS in the layouts of v_mfma_f32_32x32x2_f32, and
// the merge of a workgroup's accumulators.
#pragma once

#include "mf_common.h"

namespace mf {

// One unit: 32 consecutive rows (queries or keys) of one 128-row tile of one
// batch row, for one head.
struct F32Unit {
  int b, tile, row0, kvh, head;
};

// 32-row blocks a launch has per tile: all four, unless the one tile of a
// shorter row has fewer.  With four, most workgroups of such a row are empty; us,
// forward and backward, four -> fewer: 4096 x 8, 4/4 heads 840 and 3128 -> 234 and
// 819; 512 x 24, 16/8 heads 214 and 807 -> 120 and 300; 512 x 90 492 and 1495 ->
// 387 and 1154.  (128-row tiles took 370 and 1560, 219 and 725, 491 and 1762.)
inline int f32_blocks(int len) { return len > 96 ? 4 : (len + 31) / 32; }

// Launches `launch(order, grid)` for `items` tiles in launch order, `per_item`
// workgroups of `threads` each, in as many pieces as the limit of 2^32 - 1 threads
// per launch asks for (one piece up to 2^31 threads).
template <typename L>
inline void f32_launch(const int* order, size_t items, size_t per_item, int threads, L launch) {
  size_t piece = ((size_t)1 << 31) / (per_item * threads);
  if (piece < 1) piece = 1;
  for (size_t at = 0; at < items; at += piece)
    launch(order + at, (unsigned)(per_item * (items - at < piece ? items - at : piece)));
}

// blockIdx.x -> unit: (launch slot, 32-row block of the tile, head), the KV
// head fastest, so that with 8 KV heads each XCD's L2 holds one head's
// operands.  `div_h` is the number of heads the grid has per row block (Hq,
// or Hkv for the key side, where g_heads is 1), `div_sub` the blocks it has per
// tile (f32_blocks).  False for a block past the sequence end.
__device__ __forceinline__ bool f32_unit(const int* order, const FastDiv& div_h,
                                         const FastDiv& div_hkv, const FastDiv& div_sub,
                                         const FastDiv& div_tiles, int len, int g_heads,
                                         F32Unit& w) {
  const int blk = uniform(fast_div(blockIdx.x, div_h));
  const int h = uniform(blockIdx.x - blk * (int)div_h.d);
  const int g = uniform(fast_div(h, div_hkv));
  w.kvh = uniform(h - g * (int)div_hkv.d);
  w.head = w.kvh * g_heads + g;
  const int slot = uniform(fast_div(blk, div_sub));
  const int item = ld_const(order, slot);
  w.b = uniform(fast_div(item, div_tiles));
  w.tile = uniform(item - w.b * (int)div_tiles.d);
  w.row0 = w.tile * kTile + 32 * (blk - slot * (int)div_sub.d);
  return w.row0 < len;
}

// A 32x64 operand tile in LDS: rows of 64 floats at a pitch of 68, so that
// sixteen rows read at one 16-byte column fall on all 64 banks.  A wave loads
// its tiles from memory as whole rows (four 256-byte rows per instruction),
// keeps the next block's in registers while it works on this one's, and reads
// both operand layouts from the tile.  (Reading the row operand straight from
// memory, a 16-byte piece of 64 different lines per instruction, made every
// line cross L1 eight times: the forward, dq and dk/dv of 2 x 1499 tokens took
// 34.2, 50.5 and 59.4 us that way, 29.7, 38.8 and 46.4 this way.)
constexpr int kF32Pitch = kD + 4;
struct F32Tile {
  float x[32 * kF32Pitch];
  // the lane's dims 32 (lane / 32) + 4 j .. + 3 of row lane % 32: an operand
  // whose MFMA step st contracts dims st (lanes 0-31) and 32 + st
  __device__ __forceinline__ f32x4 row4(int lane, int j) const {
    return *reinterpret_cast<const f32x4*>(&x[(lane & 31) * kF32Pitch + 32 * (lane >> 5) + 4 * j]);
  }
  // dim 32 db + lane % 32 of row acc_row(r, lane): the transposed operand, in
  // the row order in which an accumulator's registers feed the next product
  __device__ __forceinline__ float col(int lane, int db, int r) const {
    return x[acc_row(r, lane) * kF32Pitch + 32 * db + (lane & 31)];
  }
};

// Rows r0 .. r0 + 31 as loaded: row 4 i + lane / 16, 16-byte piece lane % 16.
// `base` is wave-uniform, `stride` in bytes; offsets are 32-bit (the entry
// points reject batch rows of 4 GiB or more).  Rows past `last` re-read it, until
// f32_store drops them.
__device__ __forceinline__ void f32_load(const char* base, uint32_t stride, int r0, int last,
                                         int lane, f32x4 (&x)[8]) {
  if (r0 + 31 <= last) {
    const uint32_t off = (uint32_t)(lane >> 4) * stride + 16u * (lane & 15);
    const char* p = base + (uint32_t)r0 * stride;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      x[i] = *reinterpret_cast<const f32x4*>(p + (uint32_t)(4 * i) * stride + off);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t row = (uint32_t)min(r0 + 4 * i + (lane >> 4), last);
      x[i] = *reinterpret_cast<const f32x4*>(base + (row * stride + 16u * (lane & 15)));
    }
  }
}

// Rows `rows` and on of the block lie past the sequence end and are stored as
// zero: their probabilities are zero, and 0 * inf must not come of a row that
// was read in their place.  (Here, not at the loads, which stay in flight.)
__device__ __forceinline__ void f32_store(F32Tile& t, int lane, f32x4 (&x)[8],
                                          int rows = 32) {
  if (rows < 32) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (4 * i + (lane >> 4) >= rows) x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
    *reinterpret_cast<f32x4*>(&t.x[(4 * i + (lane >> 4)) * kF32Pitch + 4 * (lane & 15)]) = x[i];
}

// Orders a wave's own LDS writes before its later reads (and reads before
// later writes) in the compiled code; the LDS unit serves a wave in order.
__device__ __forceinline__ void wave_lds_fence() { asm volatile("" ::: "memory"); }

// A wave's 32x64 accumulator (column = row of the result) as a [row][dim] tile.
__device__ __forceinline__ void f32_put(F32Tile& t, int lane, const f32x16 (&acc)[2]) {
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[db][g4 * 4 + e];
      *reinterpret_cast<f32x4*>(
          &t.x[(lane & 31) * kF32Pitch + db * 32 + 8 * g4 + 4 * (lane >> 5)]) = v;
    }
}

__device__ __forceinline__ f32x4 f32_at(const F32Tile& t, int row, int d) {
  return *reinterpret_cast<const f32x4*>(&t.x[row * kF32Pitch + d]);
}

// Sum of the waves' tiles at (row, d .. d + 3), in wave order.
template <int W>
__device__ __forceinline__ f32x4 f32_sum(const F32Tile (&t)[W], int row, int d) {
  f32x4 x = f32_at(t[0], row, d);
#pragma unroll
  for (int w = 1; w < W; ++w) x += f32_at(t[w], row, d);
  return x;
}

}  // namespace mf
