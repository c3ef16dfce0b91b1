// The slot rows of a (token, head): what the merge of the forward's partial results and the sum of the partial dQ share.
#pragma once
#include <type_traits>
#include "attn_common.h"

namespace moba {

// The rows that such a kernel walks: every row, or with token ranges (start [n], prefix [n + 1]: range b holds the tokens
// start[b] + i for i < prefix[b + 1] - prefix[b]) those of the ranges' tokens, one range behind the other.
struct SlotRows {
  const int* start;
  const int* prefix;
  int nranges, H;
  int rows;
};
inline SlotRows slot_rows(const int* start, const int* prefix, int nranges, int H, int64_t rows) {
  return {start, prefix, nranges, H, (int)rows};
}

// The number (token * H + head) of the at-th of them, for consecutive `at` over the lanes.  A wave's rows nearly always lie in
// one range, which scalar loads find for all of them; the ranges' tokens are multiplied and `at` not divided.
__device__ __forceinline__ int slot_row(const SlotRows& p, int at) {
  if (!p.start) return at;
  const int first = __builtin_amdgcn_readfirstlane(at);
  int lo = 0, hi = p.nranges;  // prefix[lo] * H <= first < prefix[hi] * H
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (table_load(p.prefix + mid) * p.H <= first) lo = mid; else hi = mid;
  }
  int begin = table_load(p.prefix + lo), tok = table_load(p.start + lo);
  if (__any(at >= table_load(p.prefix + lo + 1) * p.H)) {
    int a = 0, b = p.nranges;
    while (b - a > 1) {
      const int mid = (a + b) >> 1;
      if (p.prefix[mid] * p.H <= at) a = mid; else b = mid;
    }
    begin = p.prefix[a];
    tok = p.start[a];
  }
  return at + (tok - begin) * p.H;
}

// Up to kMostSlotsAtOnce slots of a row (parts included) are requested at once, before the statistics and picks that say which
// are present have arrived: one round trip to memory instead of two.  (The merge of twelve takes 68 registers, seven waves to a
// SIMD; in parts 82 and five.)
// NV: slots of a row, all parts; kParts: of several parts -- slot u is slot u % K1 of part u / K1, part_rows slot rows
// behind part 0 for each; the self slot has part 0 only.
constexpr int kMostSlotsAtOnce = 12;
struct SlotPlace {
  int part, j;
};
template <bool kParts>
__device__ __forceinline__ SlotPlace slot_place(int u, int K1) {  // (u a constant, K1 uniform and at least 2 where kParts)
  if constexpr (!kParts) return {0, u};
  const int part = (u >= K1) + (u >= 2 * K1) + (u >= 3 * K1);
  return {part, u - part * K1};
}

// A row's slots as a lane of its 16 sees them: 16-byte (D = 128) or 8-byte pieces.  What the buffer holds for an absent slot may
// be anything.
template <class E, int D, int NV, bool kParts>
struct RowSlots {
  static constexpr int kPer = D / 16;
  typedef typename std::conditional<kPer == 8, u32x4, u32x2>::type bits;
  bits x[NV];
  bool present[NV];

  __device__ __forceinline__ void request(const typename E::elem* part, int row, int c8, int K1, int part_rows) {
    const char* src = (const char*)part + ((uint64_t)(uint32_t)(row * K1) * D + c8 * kPer) * 2;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const SlotPlace at = slot_place<kParts>(u, K1);
      x[u] = __builtin_nontemporal_load(reinterpret_cast<const bits*>(src + (uint64_t)(uint32_t)(at.part * part_rows + at.j) * (D * 2)));
    }
  }
  __device__ __forceinline__ void take_picks(const int* __restrict__ sel, int row, int K1) {
    const int* ps = sel + (int64_t)row * (K1 - 1) - 1;
    int pick[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const SlotPlace at = slot_place<kParts>(u, K1);
      pick[u] = at.j > 0 ? ps[at.j] : (at.part == 0 ? 0 : -1);
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) present[u] = pick[u] >= 0;
  }
  // adds w times slot u, or nothing where it does not count (absent, or without weight: an infinity there would be 0 * infinity).
  // Dropped as whole words ahead of the product, which takes fewer instructions than to drop each element's.
  __device__ __forceinline__ void add(int u, bool counts, float w, float (&acc)[kPer]) const {
    MOBA_ELEM_TYPES(E)
    typedef typename std::conditional<kPer == 8, elem8, elem4>::type vec;
    bits kept;
#pragma unroll
    for (int i = 0; i < kPer / 2; ++i) kept[i] = counts ? x[u][i] : 0u;
    const vec v = __builtin_bit_cast(vec, kept);
#pragma unroll
    for (int e = 0; e < kPer; ++e) acc[e] += w * (float)v[e];
  }
};

// Calls launch(slots, several parts) with constants for rows of at most kMostSlotsAtOnce slots; false for others.  parts: a power
// of two.
template <class Launch>
bool for_slots(int K1, int parts, Launch launch) {
  using One = std::false_type;
  using Several = std::true_type;
#define MOBA_SLOTS(NV, KIND) launch(std::integral_constant<int, NV>{}, KIND{}); return true
  if ((int64_t)K1 * parts > kMostSlotsAtOnce || (parts > 1 && K1 < 2)) return false;
  switch ((parts == 1 ? 0 : 16 * parts) + K1 * parts) {
    case 1: MOBA_SLOTS(1, One);
    case 2: MOBA_SLOTS(2, One);
    case 3: MOBA_SLOTS(3, One);
    case 4: MOBA_SLOTS(4, One);
    case 5: MOBA_SLOTS(5, One);
    case 6: MOBA_SLOTS(6, One);
    case 7: MOBA_SLOTS(7, One);
    case 8: MOBA_SLOTS(8, One);
    case 9: MOBA_SLOTS(9, One);
    case 10: MOBA_SLOTS(10, One);
    case 11: MOBA_SLOTS(11, One);
    case 12: MOBA_SLOTS(12, One);
    case 32 + 4: MOBA_SLOTS(4, Several);
    case 32 + 6: MOBA_SLOTS(6, Several);
    case 32 + 8: MOBA_SLOTS(8, Several);
    case 32 + 10: MOBA_SLOTS(10, Several);
    case 32 + 12: MOBA_SLOTS(12, Several);
    case 64 + 8: MOBA_SLOTS(8, Several);
    case 64 + 12: MOBA_SLOTS(12, Several);
  }
#undef MOBA_SLOTS
  return false;
}

}  // namespace moba
