// What the two forward attention kernels share: the parameters of a call.
#pragma once
#include "attn_common.h"

namespace moba {

template <class E>
struct FwdParams {
  const typename E::elem* q;
  const typename E::elem* k;
  const typename E::elem* v;
  typename E::elem* part_o;  // [S*H*K1, D]
  float* part_lse;  // [S*H*K1], log2 domain
  typename E::elem* out;     // [S*H, D]: where the tiles of chunks without history slots (TileTables::chunk_direct) write
  float* lse;                // [S*H], natural log
  TileTables t;
  float scale_log2;  // D^-0.5 * log2(e)
  int* queues;       // [8] tile counters, one per XCD, zero when the kernel starts
  int* redo;         // [1 + tiles] count and ids of the tiles to be computed again (see kFixedRef); count zero at the start
  int running_max;   // one workgroup per tile: track the maximum from the start
};

// Fixed-reference softmax: a row's sum of exponentials (relative to the row maximum of the tile's first key
// block) at or beyond this, or not a number, sends the tile to the form that tracks the maximum; so does an
// accumulator of the row that is not finite (a probability beyond the element type's range -- 2^16 for fp16 --
// or products with large |v| that left fp32).
constexpr float kFixedRefMaxSum = 0x1p96f;
// Whether a row's sum of exponentials left that range: infinities, NaNs and negative sums read as too large
__device__ __forceinline__ bool beyond_fixed_range(float l_tot) {
  return float_bits(l_tot) >= __builtin_bit_cast(uint32_t, kFixedRefMaxSum);
}

constexpr float kRescaleThreshold = 8.f;  // log2 units: the running max may lag the true max by this much

// One workgroup per tile: ids reach the XCDs in runs of at most an eighth of an XCD's share of the ids (log2)
inline int tile_xcd_block_log2(int64_t total) {
  int b = 0;
  while (b < 6 && (128LL << b) <= total) ++b;
  return b;
}
// one workgroup per tile (fwd_tile.hip); head_dim 128 with tile_rows 128 or 256, or 64 with 128.  Returns an error code
// of common.h.
template <class E>
int launch_fwd_tiles(const FwdParams<E>& p, int head_dim, int tile_rows, int64_t workgroups, hipStream_t st);

}  // namespace moba
