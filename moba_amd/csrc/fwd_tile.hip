// Forward attention, one workgroup per tile: the form of the forward kernel for problems of few tiles and of short
// chunks.  Tiles, slots and results are those of moba_fwd_kernel (fwd.hip); what differs is how a compute unit is
// kept busy.  There one workgroup of eight waves walks tile after tile, and the switch from one to the next (partial
// out, lookups, first copies, first products: about 14000 cycles) is paid in the open, which a tile of 2048 or 4096
// keys hides and one of 256 or 512 keys (8000 to 16000 cycles of matrix work) does not.  Here a workgroup is four
// waves (128 rows) and two of them share a compute unit (80 KiB of LDS each): one's switch runs under the other's
// matrix instructions.
//
// LDS: a ring of three K stages and two of V, 64 keys each.  At the top of key tile t a wave waits for its own copies
// of V(t) and K(t+1), issued a tile earlier; behind the barrier both are complete, nobody reads K(t-1) and V(t-1) any
// more, and their stages take K(t+2) and V(t+1).
//
// Measured, attention kernel alone: 3 x 2001 tokens, 32 heads, chunk 256, fp16: 160 -> 104 us; 20480 tokens in five
// sequences, 8 heads, chunk 512: 163 -> 130 us; 8191 tokens, 32 heads, chunk 512: 374 -> 269 us.  Beyond a few
// milliseconds the chip's power limit decides and the doubled L2 -> LDS traffic costs 3 to 8 %: those stay with
// moba_fwd_kernel (the rule stands with the caller's choice of the tile height).
//
// Heads of 64 elements (the only kernel that takes them unpadded) need half the LDS and 142 registers: three workgroups
// to a compute unit.  The exponentials weigh twice as much against the products there, so the rate in FLOP/s stays
// below that of 128 elements, but half the work is gone: 8191 tokens, 32 heads, chunk 512, whole operator: 401 us padded
// to 128, 205 us here; 131072 tokens, chunk 4096, 12 chunks: 64.8 -> 43.6 ms.
//
// Softmax: relative to the row maximum of the tile's first 32 keys (see fwd.hip); a tile in which a row leaves the
// range that is safe is computed again on the spot with a running maximum, by the same workgroup.  (FwdParams::running_max:
// with a running maximum from the start.)
#include <cstddef>
#include <type_traits>
#include "fwd_common.h"

namespace moba {

template <int D, int NW>
struct FwdTileShape {
  static constexpr int kRowBytes = 2 * D;
  static constexpr int kStage = TN * kRowBytes;     // bytes of a K or V tile
  static constexpr int kVBase = 3 * kStage;
  // D = 128: two workgroups of four waves fill the unit's 160 KiB exactly; D = 64: half of that, three fit by registers
  static constexpr int kLds = 5 * kStage;
  static constexpr int kFlags = kLds - 4 * NW;      // a word per wave; in the second V stage, free when it is used
  static constexpr int kCols = D / 8;               // 16-byte columns of a row
  static constexpr int kSlabRows = 1024 / kRowBytes;  // rows that one copy instruction of a wave brings
  static constexpr int kCopies = TN / kSlabRows / NW;  // copy instructions per wave and K or V tile
  static constexpr int kWavesPerSimd = D == 128 ? 2 : 3;
};

// The swizzle of the 16-byte columns: that of the 256-byte rows, or for 128-byte rows (two of them to the 256 bytes the
// banks span) one under which 16 consecutive rows still put the same column into 16 different places, and so do the
// 4 rows x 64 bytes of a transposed read.
template <int D>
__device__ __forceinline__ int tile_sw(int row) {
  return D == 128 ? ((row & 3) << 2) ^ ((row >> 2) & 3) : ((row & 2) << 1) | ((row >> 2) & 3);
}

// kTail: the queries are the last tokens of their sequences against a key/value cache (moba_tail_tiles below).  The
// tiles follow from sizes alone, all sequences in one launch; TileTables then holds, besides heads and strides,
//   S: query tokens per sequence, N: tiles per head of a sequence, q_shift: keys before the first query token
template <class E, int D, int NW, bool kTail>
__global__ __launch_bounds__(NW * 64, (FwdTileShape<D, NW>::kWavesPerSimd)) void fwd_tile_kernel(const FwdParams<E> p) {
  MOBA_ELEM_TYPES(E)
  using Shape = FwdTileShape<D, NW>;
  constexpr int kRows = 32 * NW, kCopies = Shape::kCopies, kStage = Shape::kStage, kRowBytes = Shape::kRowBytes;
  constexpr int kKs = D / 16, kDb = D / 32;  // matrix steps along the head dimension of S^T, row blocks of O^T
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, hh = lane >> 5;

  // ---- which tile: the parts of the history tiles (hist_bound << ks ids, the part in the low bits) and the self
  // tiles, whichever kind takes longer first: workgroups start in the order of their ids ----
  Tile t;
  int key_part = 0;
  int seq = 0, row0 = 0;  // kTail: sequence, first of its query tokens
  if constexpr (kTail) {
    const int logical = logical_tile_id(p.t.xcd_block_log2);
    if (logical >= p.t.self_total) return;
    const int sh = logical / p.t.N;
    seq = sh / p.t.H;
    row0 = (p.t.N - 1 - (logical - sh * p.t.N)) * kRows;  // (longest first)
    t.id = logical;
    t.h = sh - seq * p.t.H;
    t.row_count = min(kRows, p.t.S - row0);
    t.nkeys = p.t.q_shift + row0 + t.row_count;
    t.direct = 1;
  } else {
    int logical = logical_tile_id(p.t.xcd_block_log2);
    const int ks = p.t.key_split_log2;
    const int parts_end = p.t.hist_bound << ks;
    const int hist_part = p.t.self_first ? logical - p.t.self_total : (logical < parts_end ? logical : -1);
    if (hist_part >= parts_end) return;
    if (hist_part >= 0) {
      key_part = hist_part & ((1 << ks) - 1);
      logical = hist_part >> ks;
    } else {
      logical = p.t.hist_bound + (p.t.self_first ? logical : logical - parts_end);
    }
    if (!decode_tile_head<true>(p.t, logical, t, kRows)) return;
    if (t.base >= 0) {  // this part's share of the chunk's keys
      t.nkeys >>= ks;
      t.kv_tok0 += key_part * t.nkeys;
    }
  }
  const int h = t.h, nkeys = t.nkeys;
  const int nkt = (nkeys + TN - 1) / TN;

  // ---- K/V loader: wave w copies the 1 KiB slabs w, w + NW, ... of a tile ----
  const int64_t row_bytes = p.t.kv_tok_b;
  const uint32_t lds_base = lds_addr(smem);
  const int ld_kin = lane / Shape::kCols, ld_pc = lane % Shape::kCols;
  uint32_t ld_off[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const int key = Shape::kSlabRows * (NW * i + wave) + ld_kin;
    ld_off[i] = (uint32_t)(key * row_bytes + (ld_pc ^ tile_sw<D>(key)) * 16);
  }
  const int64_t kv_off = (kTail ? seq * p.t.kv_batch_b : kv_tok_bytes(p.t, t.kv_tok0)) + quotient_or_same(h, p.t.by_rep) * p.t.kv_head_b;
  const char* k_head = (const char*)p.k + kv_off;
  const char* v_head = (const char*)p.v + kv_off;
  auto issue = [&](const char* head, int kt, uint32_t dst) __attribute__((always_inline)) {
    const int key0 = kt * TN;
    if (key0 + TN <= nkeys) {
      const char* base = head + (int64_t)key0 * row_bytes;
#pragma unroll
      for (int i = 0; i < kCopies; ++i) async_copy16_sv(base, ld_off[i], dst + (NW * i + wave) * 1024);
    } else {
      // (keys past the end of the range: the last key again -- their scores are masked, their V rows cleared)
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        const int slab = NW * i + wave, key = Shape::kSlabRows * slab + ld_kin;
        async_copy16(head + (int64_t)min(key0 + key, nkeys - 1) * row_bytes + (ld_pc ^ tile_sw<D>(key)) * 16, dst + slab * 1024);
      }
    }
  };
  auto issue_k = [&](int kt) __attribute__((always_inline)) {
    if (kt < nkt) issue(k_head, kt, lds_base + (kt % 3) * kStage);
  };
  auto issue_v = [&](int kt) __attribute__((always_inline)) {
    if (kt < nkt) issue(v_head, kt, lds_base + Shape::kVBase + (kt & 1) * kStage);
  };
  // rows of V past the end of the key range must not reach the matrix pipe (0 * NaN): clear them
  auto scrub_v = [&](int kt) __attribute__((always_inline)) {
    const int key0 = kt * TN;
    if (key0 + TN <= nkeys) return;
    char* vdst = smem + Shape::kVBase + (kt & 1) * kStage;
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const int slab = NW * i + wave;
      if (key0 + Shape::kSlabRows * slab + ld_kin >= nkeys) *reinterpret_cast<u32x4*>(vdst + slab * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
    }
  };
  auto first_copies = [&]() __attribute__((always_inline)) {
    issue_k(0);
    issue_v(0);
    issue_k(1);
  };
  first_copies();

  // ---- this lane's row, its Q^T operand ----
  const int r = wave * 32 + n;
  const char* q_row;
  if constexpr (kTail) {
    const int row = row0 + min(r, t.row_count - 1);
    t.rh = h;
    t.dest = (seq * p.t.S + row) * p.t.H + h;
    t.limit = p.t.q_shift + row;
    t.wave_min_limit = p.t.q_shift + row0 + min(wave * 32, t.row_count - 1);
    q_row = (const char*)p.q + seq * p.t.q_batch_b + row * p.t.q_tok_b;
  } else {
    decode_tile_rows<true>(p.t, wave, r, decode_tile_row_entry(p.t, r, t), t);
    q_row = (const char*)p.q + q_tok_bytes(p.t, t.tok);
  }
  const int dest = t.dest + key_part * p.t.part_stride;  // (part 0 for a self tile)
  const int limit = t.limit;
  const int min_limit = __builtin_amdgcn_readfirstlane(t.wave_min_limit);
  const bool row_valid = r < t.row_count;
  elem8 bq[kKs];
  {
    const elem* src = reinterpret_cast<const elem*>(q_row + t.rh * p.t.q_head_b) + 8 * hh;
#pragma unroll
    for (int s8 = 0; s8 < kKs; ++s8) bq[s8] = *reinterpret_cast<const elem8*>(src + 16 * s8);
  }

  // ---- fragment addresses inside stage 0 (see fwd.hip) ----
  uint32_t koff[kKs], voffA[kDb], voffB[kDb];
  {
#pragma unroll
    for (int s8 = 0; s8 < kKs; ++s8) koff[s8] = lds_base + n * kRowBytes + (((2 * s8 + hh) ^ tile_sw<D>(n)) << 4);
    const int g16 = lane >> 4, i0 = (lane & 15) >> 2, i1 = lane & 3;
    const int v_c16 = 2 * (g16 & 1) + (i1 >> 1), v_sub = (i1 & 1) * 8;
#pragma unroll
    for (int db = 0; db < kDb; ++db) {
      const int c16 = 4 * db + v_c16, row = 4 * hh + i0;
      voffA[db] = lds_base + Shape::kVBase + row * kRowBytes + ((c16 ^ tile_sw<D>(row)) << 4) + v_sub;
      voffB[db] = lds_base + Shape::kVBase + (row + 8) * kRowBytes + ((c16 ^ tile_sw<D>(row + 8)) << 4) + v_sub;
    }
  }
  // the addresses move with the ring: K by one stage after the first half of every key tile (the second half already
  // reads the next tile's), V by one after the second
  auto k_frag = [&](int kb, int s8) __attribute__((always_inline)) { return *lds_ptr<const elem8>(koff[s8] + (uint32_t)(kb * 32 * kRowBytes)); };
  auto v_frag = [&](int kb, int j2, int db) __attribute__((always_inline)) {
    const elem4 va = lds_read_tr<elem4>(voffA[db] + (uint32_t)((32 * kb + 16 * j2) * kRowBytes));
    const elem4 vb = lds_read_tr<elem4>(voffB[db] + (uint32_t)((32 * kb + 16 * j2) * kRowBytes));
    return __builtin_shufflevector(va, vb, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  f32x16 oacc[kDb];
  float m_run, l_run;
  const float sl2 = p.scale_log2;
  auto mask_block = [&](f32x16& s, int key0) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (key0 + 8 * (e >> 2) + 4 * hh + (e & 3) > limit) s[e] = -INFINITY;
  };
  auto row_max = [&](const f32x16& s) __attribute__((always_inline)) {
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    return max_xhalf(mx) * sl2;
  };
#define MOBA_PIN(x) asm volatile("" : "+v"(x))

  // All keys of the tile; kFixed: relative to the first block's row maximum, otherwise with a running maximum.
  // Pipelined by hand over 32-key blocks like the loop of fwd.hip: S^T of the next block under the exponentials of
  // this one, O^T += V^T P^T of this one under the first exponentials of the next.
  auto all_keys = [&](auto fixed_c) __attribute__((always_inline)) {
    constexpr bool kFixed = decltype(fixed_c)::value;
#pragma unroll
    for (int db = 0; db < kDb; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[db][e] = 0.f;
    wait_vmem();
    scrub_v(0);
    __syncthreads();
    f32x16 s0, s1;
    elem8 pb[2], kpre[kKs / 2];
    {
#pragma unroll
      for (int e = 0; e < 16; ++e) s0[e] = 0.f;
#pragma unroll
      for (int s8 = 0; s8 < kKs; ++s8) s0 = mfma32(k_frag(0, s8), bq[s8], s0);
      if (31 > min_limit) mask_block(s0, 0);
      // (every row has a key in this block: key 0 of a causal tile, any key of a history tile)
      m_run = row_max(s0);
      l_run = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float pe = fast_exp2(s0[e] * sl2 - m_run);
        l_run += pe;
        pb[0][e] = (elem)pe;
      }
#pragma unroll
      for (int i = 0; i < kKs / 2; ++i) kpre[i] = k_frag(1, i);
    }
    // One step on key block kb of the tile: sc its S^T, elements 0..7 already in pb[0]; sn receives S^T of the next
    // block, block nkb of the tile koff points to; kpre holds the first four K fragments of it and receives those of
    // the block after (block 1 - nkb, after the addresses have moved if `move`).
    auto step = [&](f32x16& sc, f32x16& sn, int nkb, int next_key0, auto has_next_c, bool masked, int kb, bool pre,
                    auto move_k) __attribute__((always_inline)) {
      constexpr bool has_next = decltype(has_next_c)::value;
      elem8 ka[kKs], va[2 * kDb];
      float pf[8], rs = 0.f;
      if constexpr (has_next) {
#pragma unroll
        for (int i = 0; i < kKs / 2; ++i) ka[i] = kpre[i];
      }
#pragma unroll
      for (int s8 = 0; s8 < kKs; ++s8) {
        if constexpr (has_next) {
          if (s8 + kKs / 2 < kKs) ka[s8 + kKs / 2] = k_frag(nkb, s8 + kKs / 2);
          if (s8 == 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) sn[e] = 0.f;
          }
          sn = mfma32(ka[s8], bq[s8], sn);
        }
#pragma unroll
        for (int e = s8 * (8 / kKs); e < (s8 + 1) * (8 / kKs); ++e) {
          pf[e] = fast_exp2(sc[8 + e] * sl2 - m_run);
          if (e > 0) rs += pf[e - 1];
          MOBA_PIN(pf[e]);
          MOBA_PIN(rs);
        }
        if (s8 >= kKs / 2 && s8 < kKs / 2 + 2) {  // half of the first V fragments each
#pragma unroll
          for (int db = (s8 - kKs / 2) * (kDb / 2); db < (s8 - kKs / 2 + 1) * (kDb / 2); ++db) va[db] = v_frag(kb, 0, db);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      move_k();
      l_run += rs + pf[7];
#pragma unroll
      for (int e = 0; e < 8; ++e) pb[1][e] = (elem)pf[e];
      if constexpr (has_next) {
        if (masked) mask_block(sn, next_key0);
      }
      float pg[8], rn = 0.f;
#pragma unroll
      for (int k = 0; k < 2 * kDb; ++k) {
        if (k < kDb) va[k + kDb] = v_frag(kb, 1, k);
        if (k >= kDb && pre) {
#pragma unroll
          for (int i = (k - kDb) * kKs / (2 * kDb); i < (k - kDb + 1) * kKs / (2 * kDb); ++i) kpre[i] = k_frag(1 - nkb, i);
        }
        oacc[k % kDb] = mfma32(va[k], pb[k / kDb], oacc[k % kDb]);
        if constexpr (has_next && kFixed) {
          // the eight exponentials spread over the slots behind the first, which is left to the last S^T product's result
          const int e0 = k == 0 ? 0 : (k == 1 ? 0 : (kDb == 4 ? k : 3 * k - 4));
          const int e1 = k == 0 ? 0 : (k == 1 ? 2 : (kDb == 4 ? k + 1 : 3 * k - 1));
#pragma unroll
          for (int e = e0; e < e1; ++e) {
            pg[e] = fast_exp2(sn[e] * sl2 - m_run);
            MOBA_PIN(pg[e]);
            if (e > 1) {
              rn = e == 2 ? pg[0] + pg[1] : rn + pg[e - 1];
              MOBA_PIN(rn);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (has_next && !kFixed) {  // the rare form: no slots
        const float mx = row_max(sn);
        const float m_new = mx > m_run + kRescaleThreshold ? mx : m_run;
        const float alpha = fast_exp2(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < kDb; ++db)
#pragma unroll
          for (int e = 0; e < 16; ++e) oacc[db][e] *= alpha;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pg[e] = fast_exp2(sn[e] * sl2 - m_run);
          if (e < 7) rn += pg[e];
        }
      }
      if constexpr (has_next) {
        l_run += rn + pg[7];
#pragma unroll
        for (int e = 0; e < 8; ++e) pb[0][e] = (elem)pg[e];
      }
    };
    int kstage = 0;
    auto move_k = [&]() __attribute__((always_inline)) {
      const uint32_t d = kstage == 2 ? (uint32_t)(-2 * kStage) : (uint32_t)kStage;
      kstage = kstage == 2 ? 0 : kstage + 1;
#pragma unroll
      for (int s8 = 0; s8 < kKs; ++s8) koff[s8] += d;
    };
    auto stay = [] __attribute__((always_inline)) {};
    auto tile_body = [&](int it, auto more_c) __attribute__((always_inline)) {
      constexpr bool more = decltype(more_c)::value;  // a key tile follows this one
      const int key0 = it * TN;
      if (it > 0) {
        wait_vmem();
        scrub_v(it);
        __syncthreads();
      }
      if constexpr (more) {
        issue_k(it + 2);
        issue_v(it + 1);
      }
      step(s0, s1, 1, key0 + 32, std::true_type{}, key0 + 63 > min_limit, 0, more, move_k);
      step(s1, s0, 0, key0 + TN, more_c, more && key0 + TN + 31 > min_limit, 1, more, stay);
      const uint32_t d = (it & 1) ? (uint32_t)(-kStage) : (uint32_t)kStage;
#pragma unroll
      for (int db = 0; db < kDb; ++db) {
        voffA[db] += d;
        voffB[db] += d;
      }
    };
    int it = 0;
    for (; it + 1 < nkt; ++it) tile_body(it, std::true_type{});
    tile_body(it, std::false_type{});
    __syncthreads();  // every wave has read its last fragments: the stages are free
  };
#undef MOBA_PIN

  float l_tot = 0.f;
  int again = p.running_max;
  if (!again) {
    all_keys(std::true_type{});
    l_tot = sum_xhalf(l_run);
    const bool bad = row_valid && (beyond_fixed_range(l_tot) || any_not_finite(oacc));
    volatile int* flags = reinterpret_cast<volatile int*>(smem + Shape::kFlags);
    const bool any_bad = __any(bad);
    if (lane == 0) flags[wave] = any_bad ? 1 : 0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) again |= flags[w];
    again = __builtin_amdgcn_readfirstlane(again);
    if (again) {
      __syncthreads();  // (every wave has read the flags)
      // back to stage 0: nkt tiles moved K by nkt stages, V by nkt
      const uint32_t dk = (uint32_t)((nkt % 3) * kStage), dv = (uint32_t)((nkt & 1) * kStage);
#pragma unroll
      for (int s8 = 0; s8 < kKs; ++s8) koff[s8] -= dk;
#pragma unroll
      for (int db = 0; db < kDb; ++db) {
        voffA[db] -= dv;
        voffB[db] -= dv;
      }
      first_copies();
      if (p.redo && tid == 0) {  // (listed for a caller that asks which tiles these were)
        const int at = __hip_atomic_fetch_add(p.redo, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (every part of a cut tile counts: more of them than the array has entries are counted only)
        if (at < p.t.hist_bound + p.t.self_total) p.redo[1 + at] = t.id;
      }
    }
  }
  if (again) {
    all_keys(std::false_type{});
    l_tot = sum_xhalf(l_run);
  }

  // ---- normalise, write: through 4 KiB of LDS per wave, half a row at a time, so that the rows leave as 128-byte
  // pieces, eight rows per store instruction (see fwd.hip) ----
  {
    const float inv = 1.f / l_tot;
    char* stage = smem + wave * 4096;
    char* wrow = stage + n * 128 + 8 * hh;
    const int wsw = (n >> 1) & 7;
    elem* const o_base = t.direct ? p.out : p.part_o;
    if (!kTail && row_valid && hh == 0) {
      const float l2 = m_run + fast_log2(l_tot);
      if (t.direct) p.lse[dest] = l2 * 0.6931471805599453f;
      else p.part_lse[dest] = l2;
    }
    const int c16 = lane & 7;
    const int rows_here = t.row_count - wave * 32;
    int d4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d4[i] = __shfl(dest, 8 * i + (lane >> 3), 64);
#pragma unroll
    for (int half = 0; half < D / 64; ++half) {
#pragma unroll
      for (int d2 = 0; d2 < 2; ++d2)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int db = 2 * half + d2;
          u32x2 w;
          w[0] = pack2<E>(oacc[db][4 * g + 0] * inv, oacc[db][4 * g + 1] * inv);
          w[1] = pack2<E>(oacc[db][4 * g + 2] * inv, oacc[db][4 * g + 3] * inv);
          *reinterpret_cast<u32x2*>(wrow + (((4 * d2 + g) ^ wsw) << 4)) = w;
        }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * i + (lane >> 3);
        const u32x4 x = *reinterpret_cast<const u32x4*>(stage + row * 128 + ((c16 ^ ((row >> 1) & 7)) << 4));
        if (row < rows_here) *reinterpret_cast<u32x4*>(o_base + (int64_t)d4[i] * D + 64 * half + c16 * 8) = x;
      }
    }
  }
}

template <class E, int D, int NW, bool kTail>
static int launch(const FwdParams<E>& p, int64_t workgroups, hipStream_t st) {
  using Shape = FwdTileShape<D, NW>;
  static bool allowed[kMaxDevices];
  if (!allow_dynamic_lds((const void*)fwd_tile_kernel<E, D, NW, kTail>, Shape::kLds, allowed)) return MOBA_ERR_LAUNCH;
  hipLaunchKernelGGL((fwd_tile_kernel<E, D, NW, kTail>), dim3((unsigned)workgroups), dim3(NW * 64), Shape::kLds, st, p);
  return MOBA_OK;
}

template <class E>
int launch_fwd_tiles(const FwdParams<E>& p, int head_dim, int tile_rows, int64_t workgroups, hipStream_t st) {
  if (head_dim == 64) return launch<E, 64, 4, false>(p, workgroups, st);
  return tile_rows == 128 ? launch<E, 128, 4, false>(p, workgroups, st) : launch<E, 128, 8, false>(p, workgroups, st);
}
template int launch_fwd_tiles<Bf16>(const FwdParams<Bf16>&, int, int, int64_t, hipStream_t);
template int launch_fwd_tiles<F16>(const FwdParams<F16>&, int, int, int64_t, hipStream_t);

// Rows per tile of moba_tail_tiles, for `row_blocks` blocks of 128 query tokens in all or `tall` of 256.  Tall tiles move half
// the bytes from L2 to LDS, but one fills a compute unit and a short one half of it.  In units of a full round of tall
// tiles (one per unit), measured at 32 and 16 heads, 40000 keys: a full round of short ones (two per unit) 1.035, up to
// one per unit 0.49 to 0.58, above that 0.82 to 1.035; up to half a round of tall ones 0.71, the rest 0.75 to 1.
//   2048 tokens, 32 heads, 34816 keys: 1.04 ms short, 0.975 tall; 4 sequences x 1100 tokens, 16 heads, 40000 keys: 1.60
//   short, 1.88 tall; 2048 tokens, 8 heads, 40000 keys: 0.54 short, 0.79 tall
static int tail_tile_rows(int64_t blocks, int64_t tall, int cus) {
  auto cost = [](int64_t n, int64_t round, double full, double few, double low) {
    const int64_t rest = n % round;
    const double part = (double)rest / (double)round;
    return full * (double)(n / round) + (rest == 0 ? 0. : (2 * rest <= round ? few : low + (full - low) * part));
  };
  return cost(blocks, 2 * (int64_t)cus, 1.035, 0.55, 0.6) < cost(tall, cus, 1., 0.71, 0.5) ? 128 : 256;
}

template <class E>
static int launch_tail_tiles(const void* q, const void* k, const void* v, void* out, const TileTables& t, float scale,
                             int running_max, int64_t workgroups, int tile_rows, hipStream_t st) {
  LaunchCheck launch_check;
  FwdParams<E> p = {};
  p.q = (const typename E::elem*)q; p.k = (const typename E::elem*)k; p.v = (const typename E::elem*)v;
  p.out = (typename E::elem*)out;
  p.t = t;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.running_max = running_max;
  const int rc = tile_rows == 128 ? launch<E, 128, 4, true>(p, workgroups, st) : launch<E, 128, 8, true>(p, workgroups, st);
  return rc != MOBA_OK ? rc : launch_check.result();
}

}  // namespace moba

using namespace moba;

// The last nq tokens of B sequences against their keys and values, on the causal tiles of fwd_tile_kernel: token j sees
// keys 0 .. Skv - nq + j.  q, k and v are read in place, all sequences in one launch: one launch per sequence left most
// of the chip idle whenever heads * nq / 256 was below the number of compute units, and copied q and the result.
// 4 sequences x 1024 tokens, 8 heads, 9000 keys: 836 -> 166 us; 4 x 2048, 32 heads, 9000 keys: 1771 -> 993 us; one of 2048
// tokens, 32 heads, 34816 keys: 1018 -> 961 us (bound by the products: 1.18 PFLOP/s).
extern "C" int moba_tail_tiles(const void* q, const void* k, const void* v, void* out, int B, int H, int Hkv, int nq,
                               int Skv, int D, const int64_t* strides, float scale, int dtype, int running_max,
                               void* stream) {
  if (!q || !k || !v || !out || !strides) return MOBA_ERR_ARG;
  if (B <= 0 || H <= 0 || Hkv <= 0 || nq <= 0 || nq > Skv || H % Hkv != 0 || !(scale > 0.f)) return MOBA_ERR_ARG;
  if (D != kHeadDim || (dtype != MOBA_DTYPE_BF16 && dtype != MOBA_DTYPE_F16)) return MOBA_ERR_UNSUPPORTED;
  if (((uintptr_t)q & 15) || ((uintptr_t)k & 15) || ((uintptr_t)v & 15) || ((uintptr_t)out & 15)) return MOBA_ERR_ARG;
  for (int i = 0; i < 6; ++i)
    if (strides[i] < 0 || (strides[i] & 7)) return MOBA_ERR_ARG;  // 16-byte accesses
  if (strides[5] > (1 << 23)) return MOBA_ERR_ARG;                // (a key tile's byte offsets fit 31 bits)
  const int64_t heads = (int64_t)B * H;
  if (heads >= 0x7fffffffLL || heads * nq >= 0x7fffffffLL) return MOBA_ERR_LIMIT;
  const int cus = resident_compute_units();
  if (cus <= 0) return MOBA_ERR_LAUNCH;
  const int tile_rows = tail_tile_rows(heads * (((int64_t)nq + 127) / 128), heads * (((int64_t)nq + 255) / 256), cus);
  const int64_t tiles = ((int64_t)nq + tile_rows - 1) / tile_rows, total = heads * tiles;
  TileTables t = {};
  t.S = nq; t.N = (int)tiles; t.q_shift = Skv - nq; t.self_total = (int)total;
  t.H = H; t.Hkv = Hkv; t.rep = H / Hkv; t.by_rep = divisor_or_one(t.rep); t.K1 = 1;
  t.q_batch_b = strides[0] * 2; t.q_head_b = strides[1] * 2; t.q_tok_b = strides[2] * 2;
  t.kv_batch_b = strides[3] * 2; t.kv_head_b = strides[4] * 2; t.kv_tok_b = strides[5] * 2;
  t.xcd_block_log2 = tile_xcd_block_log2(total);
  const int64_t run = 8LL << t.xcd_block_log2, workgroups = (total + run - 1) / run * run;
  if (workgroups >= 0x7fffffffLL) return MOBA_ERR_LIMIT;
  hipStream_t st = (hipStream_t)stream;
  running_max = running_max != 0;
  return dtype == MOBA_DTYPE_F16
             ? launch_tail_tiles<F16>(q, k, v, out, t, scale, running_max, workgroups, tile_rows, st)
             : launch_tail_tiles<Bf16>(q, k, v, out, t, scale, running_max, workgroups, tile_rows, st);
}
