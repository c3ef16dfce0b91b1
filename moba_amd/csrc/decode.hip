// Decode attention: the last `nq` tokens of every sequence against its key/value cache, the branch of the
// reference adapter that calls flash_attn_func with few query tokens (moba/wrapper.py:76-82).  Token j of the nq
// sees the keys up to its own position Skv - nq + j; grouped-query heads are handled in place; the softmax scale is
// the caller's.
//
// HBM-bound: K and V of the cache are to be read once.  The nq * rep query rows that share a key/value head are
// columns of a matrix product (S^T = K Q^T, O^T += V^T P^T with v_mfma_f32_32x32x16), so that up to 32 of them take one
// pass over the cache: a kernel that gives every row its own dot products is bound by the vector unit from a handful of
// rows on, and one that runs once per new token reads the cache that often.  A workgroup takes a range of the keys
// (a split); its four waves take different keys of it, or different blocks of 32 rows once there are more than 32 (two or
// four waves then copy the same keys, from L2); beyond 128 rows further workgroups walk the same range, a pass each.
// A wave copies its own K and V blocks of 32 keys global -> LDS (two stages of 16 KiB, no barrier: the wait for a
// block counts the wave's own copies) while it computes the block before: 64 to 128 KiB per compute unit in flight,
// where about 40 KiB cover the latency at the full rate.  One workgroup per compute unit (128 KiB of LDS); the
// splits are chosen so that the workgroups come out just below a multiple of the units.  Where the sequences alone are more than
// the units, short caches take workgroups of two waves or one, two or five to a unit (tail_split).
// Keys that one wave reads alone (up to 32 rows) are copied past the caches: 1 x 65536 keys, 64 heads: 368 us without, 314
// with (6.8 TB/s); keys that several waves or workgroups read are not: 40000 keys, 128 rows: 69.4 us without, 75.6 with.
//
// Measured (32 query heads on 8): 131072 keys, one token: 84 us a call = 6.4 TB/s (108 with a vector-unit kernel of 128
// splits); 16 x 8191 keys: 84 us = 6.4 TB/s (102); 4 x 20000 keys, 5 tokens: 60 us (348, once per token).
// Beyond 128 rows per key/value head it is bound by its own instruction chain (one wave per SIMD), 0.45 PFLOP/s.
//
// Precision: the scores' products are exact, their sums fp32.  A probability is fed to the second product as the sum
// of three elements (its rounded value, the rounded rest, and the rest of that), which hold all 24 bits of it: the matrix
// pipe has the time, and one element alone would double the error of the result.  Beyond kTailExactTokens tokens two
// elements (16 or 22 bits): there the products are the bound, and the other kernel for such calls, the causal tiles,
// rounds to one.
//
// Values that are not finite: a probability of 0 for a key that a row does not see still meets the key's value in the
// products, and 0 * Inf and the split probabilities' parts times Inf are NaN; a maximum that lags overflows for values near
// the end of bf16's range.  A wave whose accumulators are not finite at the end goes through its keys again one by one,
// in fp32, relative to the exact maximum, every row with the keys it sees only.
//
//   tail_partial_kernel   part_o[row, split, :] (normalised, fp32), part_lse (log2 domain); one split: out itself
//   tail_merge_kernel     out[row, :]
#include "attn_common.h"

namespace moba {

constexpr int kTailKeys = 32;                                 // keys a wave handles per step
constexpr int kTailTile = kTailKeys * kHeadDim * 2;           // bytes of its K (or V) block
constexpr int kTailWaveLds = 4 * kTailTile;                   // two stages of K and V
constexpr int kTailRedRow = kHeadDim + 4;                     // floats per row when the waves' sums meet in LDS
constexpr int kTailRedStats = 32 * kTailRedRow * 4;           // times the waves: byte offset of their 32 maxima each, then sums
static_assert(kTailRedStats + 2 * 32 * 4 <= kTailWaveLds, "the waves' sums fit the stages");
constexpr int kTailMaxSplits = 128;
constexpr int kTailExactTokens = 16;  // up to so many new tokens the probabilities keep their 24 bits

// the results and the scratch may lie wherever their elements can
typedef u32x2 u32x2_any __attribute__((aligned(2)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef float f32x2_any __attribute__((ext_vector_type(2), aligned(4)));

template <class E>
struct TailParams {
  const typename E::elem* q;
  const typename E::elem* k;
  const typename E::elem* v;
  typename E::elem* out;  // [B, nq, H, D]
  float* part_o;          // [B*nq*H, nsplit, D]
  float* part_lse;        // [B*nq*H, nsplit]
  int64_t q_stride_b, q_stride_h, q_stride_t, kv_stride_b, kv_stride_h;  // elements
  int Hkv, rep, Skv, nq;
  int wr_log2;            // log2 of the row blocks of a workgroup (its other waves split the keys)
  int keys_per_split, nsplit;
  float scale_log2;
};

// fp16 probabilities are kept 2^7 times larger (the running maximum may lag by 2^8: they stay below 2^15), so that
// those far below the maximum stay above the type's smallest number; the factor cancels
template <class E> struct TailShift { static constexpr float value = 0.f; };
template <> struct TailShift<F16> { static constexpr float value = 7.f; };
constexpr float kTailMaxLag = 8.f;
constexpr float kTailNoMax = -3e38f;  // before the first visible key (finite: exp2(m - m_new) stays defined)

// kOnce: one workgroup and one wave reads a key's rows (up to 32 query rows per key/value head): they pass the caches by
// (Held to 256 registers, though its LDS lets one wave per SIMD run: with all 512 the compiler keeps the sums in accumulation
// registers and moves all of them for every rescale and for the end; partial kernel at 4097 keys: 9.4 us so, 8.9 held.)
// NW: waves of a workgroup; fewer than four go with kOnce
template <class E, bool kOnce, int NW>
__global__ __launch_bounds__(64 * NW, 2) void tail_partial_kernel(const TailParams<E> p) {
  MOBA_ELEM_TYPES(E)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, hh = lane >> 5;
  const int split = blockIdx.x, b = blockIdx.z;
  const int group = blockIdx.y / p.Hkv, hkv = blockIdx.y - group * p.Hkv;
  const int wr_n = 1 << p.wr_log2, wk_n = NW >> p.wr_log2;
  const int wr = wave & (wr_n - 1), wk = wave >> p.wr_log2;
  const int rows = p.nq * p.rep;
  const int row0 = (group * wr_n + wr) * 32;
  const int row = min(row0 + n, rows - 1);  // (rows past the last repeat it and are not written)
  const int j = row / p.rep, g = row - j * p.rep;
  const int key_lo = split * p.keys_per_split, key_hi = min(p.Skv, key_lo + p.keys_per_split);
  const int limit = min(p.Skv - p.nq + j, key_hi - 1);          // the row's last visible key in this split
  const int first_masked = min(p.Skv - p.nq, key_hi - 1);       // keys up to here are visible to every row
  const int nblk = (key_hi - key_lo + kTailKeys - 1) / kTailKeys;
  const int mine = row0 < rows ? (nblk - wk + wk_n - 1) / wk_n : 0;  // blocks wk, wk + wk_n, ... are this wave's

  // K/V loader: one instruction copies 4 keys x 256 bytes; lane i lands at 16*i, so it picks the global column whose
  // swizzled place that is
  const uint32_t lds_base = lds_addr(smem) + wave * kTailWaveLds;
  const int ld_kin = lane >> 4, ld_pc = lane & 15;
  uint32_t ld_off[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) ld_off[i] = (4 * i + ld_kin) * 256 + sw_col16(4 * i + ld_kin, ld_pc) * 16;
  const char* k_head = (const char*)(p.k + b * p.kv_stride_b + (int64_t)hkv * p.kv_stride_h);
  const char* v_head = (const char*)(p.v + b * p.kv_stride_b + (int64_t)hkv * p.kv_stride_h);
  auto issue = [&](int it, int stage) __attribute__((always_inline)) {
    const int key0 = key_lo + (wk + it * wk_n) * kTailKeys;
    const uint32_t kdst = lds_base + stage * 2 * kTailTile, vdst = kdst + kTailTile;
    if (key0 + kTailKeys <= key_hi) {
      const int64_t off = (int64_t)key0 * 256;
#pragma unroll
      for (int i = 0; i < 8; ++i) async_copy16_sv<kOnce>(k_head + off, ld_off[i], kdst + i * 1024);
#pragma unroll
      for (int i = 0; i < 8; ++i) async_copy16_sv<kOnce>(v_head + off, ld_off[i], vdst + i * 1024);
    } else {  // (keys past the end: the last key again; their scores are masked)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int64_t off = (int64_t)min(key0 + 4 * i + ld_kin, key_hi - 1) * 256 + (ld_off[i] & 255);
        async_copy16<kOnce>(k_head + off, kdst + i * 1024);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int64_t off = (int64_t)min(key0 + 4 * i + ld_kin, key_hi - 1) * 256 + (ld_off[i] & 255);
        async_copy16<kOnce>(v_head + off, vdst + i * 1024);
      }
    }
  };

  // Q^T operand: lane (n, hh) holds q[row n][16*s8 + 8*hh .. +7]
  elem8 bq[8];
  {
    const elem* src = p.q + b * p.q_stride_b + (int64_t)(hkv * p.rep + g) * p.q_stride_h + j * p.q_stride_t + 8 * hh;
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) bq[s8] = *reinterpret_cast<const elem8*>(src + 16 * s8);
  }
  if (mine > 0) issue(0, 0);
  if (mine > 1) issue(1, 1);

  // fragment addresses inside stage 0 (see the forward kernel)
  uint32_t koff[8], voffA[4], voffB[4];
  {
    const int k_sw = ((n & 3) << 2) ^ ((n >> 2) & 3);
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) koff[s8] = lds_base + n * 256 + (((2 * s8 + hh) ^ k_sw) << 4);
    const int g16 = lane >> 4, i0 = (lane & 15) >> 2, i1 = lane & 3;
    const int v_c16 = 2 * (g16 & 1) + (i1 >> 1), v_sub = (i1 & 1) * 8;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const int c16 = 4 * db + v_c16;
      voffA[db] = lds_base + kTailTile + (4 * hh + i0) * 256 + ((c16 ^ (i0 << 2) ^ hh) << 4) + v_sub;
      voffB[db] = lds_base + kTailTile + (4 * hh + i0 + 8) * 256 + ((c16 ^ (i0 << 2) ^ (hh + 2)) << 4) + v_sub;
    }
  }

  f32x16 oacc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[db][e] = 0.f;
  float m_run = kTailNoMax, l_run = 0.f;

  for (int it = 0; it < mine; ++it) {
    const uint32_t st = (it & 1) * 2 * kTailTile;
    // this block's 16 copies have landed (the next block's 16 may still be in flight)
    if (it + 1 < mine) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
    elem8 ka[8];
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) ka[s8] = *lds_ptr<const elem8>(koff[s8] + st);
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) s = mfma32(ka[s8], bq[s8], s);
    // the V^T fragments travel while the softmax runs
    elem8 va[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j2 = i >> 2, db = i & 3;
      const elem4 a = lds_read_tr<elem4>(voffA[db] + st + 16 * j2 * 256);
      const elem4 c = lds_read_tr<elem4>(voffB[db] + st + 16 * j2 * 256);
      va[i] = __builtin_shufflevector(a, c, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    const int key0 = key_lo + (wk + it * wk_n) * kTailKeys;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] *= p.scale_log2;
    if (key0 + kTailKeys - 1 > first_masked) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (key0 + 8 * (e >> 2) + 4 * hh + (e & 3) > limit) s[e] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    mx = max_xhalf(mx);
    if (__any(mx > m_run + kTailMaxLag)) {  // rare once the maximum has settled
      const float m_new = mx > m_run + kTailMaxLag ? mx : m_run;
      const float alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[db][e] *= alpha;
    }
    const float ref = m_run - TailShift<E>::value;
    elem8 hi[2], lo[2];
    float rest[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float pe = fast_exp2(s[e] - ref);
      l_run += pe;
      const elem h = (elem)pe;
      const float r = pe - (float)h;
      const elem l = (elem)r;
      hi[e >> 3][e & 7] = h;
      lo[e >> 3][e & 7] = l;
      rest[e] = r - (float)l;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) oacc[i & 3] = mfma32(va[i], hi[i >> 2], oacc[i & 3]);
#pragma unroll
    for (int i = 0; i < 8; ++i) oacc[i & 3] = mfma32(va[i], lo[i >> 2], oacc[i & 3]);
    if (p.nq <= kTailExactTokens) {
      elem8 last[2];
#pragma unroll
      for (int e = 0; e < 16; ++e) last[e >> 3][e & 7] = (elem)rest[e];
#pragma unroll
      for (int i = 0; i < 8; ++i) oacc[i & 3] = mfma32(va[i], last[i >> 2], oacc[i & 3]);
    }
    if (it + 2 < mine) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every fragment of this stage is in registers
      issue(it + 2, it & 1);
    }
  }
  if (__builtin_expect(__any(any_not_finite(oacc)), 0)) {  // (never for values of ordinary size)
    auto each_key = [&](auto use) __attribute__((always_inline)) {
      for (int it = 0; it < mine; ++it) {
        const int key0 = key_lo + (wk + it * wk_n) * kTailKeys, key1 = min(key0 + kTailKeys, key_hi);
        for (int key = key0; key < key1; ++key) {
          const elem* kr = (const elem*)(k_head + (int64_t)key * 256) + 8 * hh;
          float d = 0.f;
#pragma unroll
          for (int s8 = 0; s8 < 8; ++s8) {
            const elem8 x = *reinterpret_cast<const elem8*>(kr + 16 * s8);
#pragma unroll
            for (int e = 0; e < 8; ++e) d += (float)bq[s8][e] * (float)x[e];
          }
          const float sc = sum_xhalf(d) * p.scale_log2;
          if (key <= limit) use(key, sc);
        }
      }
    };
    m_run = kTailNoMax;
    each_key([&](int, float sc) __attribute__((always_inline)) { m_run = fmaxf(m_run, sc); });
    const float ref = m_run - TailShift<E>::value;
    float l = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[db][e] = 0.f;
    each_key([&](int key, float sc) __attribute__((always_inline)) {
      const float pe = fast_exp2(sc - ref);
      l += pe;
      const elem* vr = (const elem*)(v_head + (int64_t)key * 256) + 4 * hh;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const elem4 x = *reinterpret_cast<const elem4*>(vr + 8 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) oacc[i >> 2][4 * (i & 3) + e] += pe * (float)x[e];
      }
    });
    l_run = hh == 0 ? l : 0.f;
  }
  l_run = sum_xhalf(l_run);

  // The waves that hold the same rows meet in LDS.  Element e of lane (n, hh) is O[row n][32*db + 8*(e/4) + 4*hh + e%4].
  __syncthreads();  // every wave has read its last fragments
  float* red = reinterpret_cast<float*>(smem);
  float* red_m = reinterpret_cast<float*>(smem + NW * kTailRedStats);
  float* red_l = red_m + NW * 32;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      *reinterpret_cast<f32x4*>(red + (wave * 32 + n) * kTailRedRow + 32 * db + 8 * g4 + 4 * hh) =
          f32x4{oacc[db][4 * g4], oacc[db][4 * g4 + 1], oacc[db][4 * g4 + 2], oacc[db][4 * g4 + 3]};
  if (hh == 0) {
    red_m[wave * 32 + n] = m_run;
    red_l[wave * 32 + n] = l_run;
  }
  __syncthreads();
  const int rows_here = min(32 * wr_n, rows - group * wr_n * 32);
  for (int i = tid; i < rows_here * 32; i += 64 * NW) {
    const int rr = i >> 5, d = (i & 31) * 4;      // row of the workgroup, dimension
    const int w0 = rr >> 5, nn = rr & 31;         // its row block (= its first wave), its row in there
    float mm = red_m[w0 * 32 + nn];
    for (int w = 1; w < wk_n; ++w) mm = fmaxf(mm, red_m[(w0 + (w << p.wr_log2)) * 32 + nn]);
    float ll = 0.f;
    f32x4 oo = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < wk_n; ++w) {
      const int at = (w0 + (w << p.wr_log2)) * 32 + nn;
      const float a = fast_exp2(red_m[at] - mm);
      ll += red_l[at] * a;
      const f32x4 x = *reinterpret_cast<const f32x4*>(red + at * kTailRedRow + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) oo[e] += x[e] * a;
    }
    const int rg = group * wr_n * 32 + rr;
    const int jj = rg / p.rep, gg = rg - jj * p.rep;
    const int64_t orow = ((int64_t)b * p.nq + jj) * (p.Hkv * p.rep) + hkv * p.rep + gg;
    // (a row may see no key of its split: the causal limit; never without another split that it does see)
    const float inv = ll > 0.f || p.nsplit == 1 ? 1.f / ll : 0.f;
    if (p.nsplit == 1) {
      u32x2 w;
      w[0] = pack2<E>(oo[0] * inv, oo[1] * inv);
      w[1] = pack2<E>(oo[2] * inv, oo[3] * inv);
      *reinterpret_cast<u32x2_any*>(p.out + orow * kHeadDim + d) = w;
    } else {
      const int64_t prow = orow * p.nsplit + split;
      *reinterpret_cast<f32x4_any*>(p.part_o + prow * kHeadDim + d) =
          f32x4{oo[0] * inv, oo[1] * inv, oo[2] * inv, oo[3] * inv};
      if (d == 0) p.part_lse[prow] = ll > 0.f ? mm - TailShift<E>::value + fast_log2(ll) : -INFINITY;
    }
  }
}

// One workgroup per output row: four waves take a quarter of the splits each, a lane owns two head dimensions; the
// four partial sums meet in LDS.
template <class E>
__global__ __launch_bounds__(256) void tail_merge_kernel(const float* __restrict__ part_o,
                                                         const float* __restrict__ part_lse,
                                                         typename E::elem* __restrict__ out, int nsplit) {
  typedef typename E::elem elem;
  __shared__ float red[4][kHeadDim];
  __shared__ float red_l[4];
  const int64_t row = blockIdx.x;  // (b * nq + j) * H + h
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* pl = part_lse + row * nsplit;
  float mm = -INFINITY;
  for (int i = lane; i < nsplit; i += 64) mm = fmaxf(mm, pl[i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o, 64));
  float ll = 0.f, o0 = 0.f, o1 = 0.f;
  const float* po = part_o + row * nsplit * kHeadDim + 2 * lane;
  for (int i = wave; i < nsplit; i += 4) {
    const float w = fast_exp2(pl[i] - mm);
    const f32x2_any x = *reinterpret_cast<const f32x2_any*>(po + (int64_t)i * kHeadDim);
    ll += w;
    o0 += w * x.x;
    o1 += w * x.y;
  }
  red[wave][2 * lane] = o0;
  red[wave][2 * lane + 1] = o1;
  if (lane == 0) red_l[wave] = ll;
  __syncthreads();
  if (threadIdx.x < kHeadDim) {
    const int d = threadIdx.x;
    const float l4 = red_l[0] + red_l[1] + red_l[2] + red_l[3];
    out[row * kHeadDim + d] = (elem)((red[0][d] + red[1][d] + red[2][d] + red[3][d]) / l4);
  }
}

}  // namespace moba

using namespace moba;

struct TailSplit {
  int wr_log2, groups, keys_per_split, nsplit;  // groups: workgroups per (sequence, key/value head, split)
  int waves;                                    // of a workgroup: 4 or 1
};

// How the work is cut: row blocks over the waves of a workgroup, then the keys over workgroups.
//
// Up to 32 rows a workgroup of four, two or one waves would do, of which a compute unit holds one, two or five: small ones
// run their starts (first copies) and ends (sums through LDS) under the copies of the others, where there are
// sequences enough to fill the chip with them, and few large ones leave least to merge where there are not.  A
// step (kTailKeys keys per wave) takes what the waves beside it on the unit leave it of latency, or of the chip's
// bandwidth if that is longer, and every round of workgroups a start and an end; the cut is the one that comes out shortest.  The
// numbers, hundredths of a microsecond up to a common factor, rank 25 cuts at 230 sizes to within 1 % of the best one on
// average.  Four waves each whatever the size / so, key/value heads of all sequences x keys: 2000 x 8, 64: 239 / 84 us; 1024, 300:
// 41 / 29; 8192, 128: 155 / 86; 1024, 600: 60 / 52; 320, 1000: 41 / 34; 200, 2500: 55 / 44.  Beyond 4096 keys a start and an
// end weigh little and four waves keep pace better (1300 x 6000: 591 us, 611 with two).
static TailSplit tail_split(int B, int Hkv, int rows, int Skv) {
  TailSplit t;
  t.wr_log2 = rows <= 32 ? 0 : (rows <= 64 ? 1 : 2);
  t.groups = (rows + (32 << t.wr_log2) - 1) / (32 << t.wr_log2);
  const bool once = t.wr_log2 == 0;
  const int64_t wgs = (int64_t)B * Hkv * t.groups;
  int cus = compute_units();
  if (cus <= 0) cus = 256;
  const bool many = once && wgs > cus && Skv <= 4096;
  // (one round, and what rounds the last one of several off: more splits are starts and ends for nothing)
  const int most = once ? (int)(cus / wgs) + 8 : kTailMaxSplits;
  int64_t best = -1;
  for (int waves = 4; waves >= (many ? 1 : 4); waves >>= 1) {
    const int unit = kTailKeys * (waves >> t.wr_log2);
    const int steps = (Skv + unit - 1) / unit;
    const int slots = cus * (waves == 1 ? 5 : 4 / waves);
    auto step_time = [&](int workgroups) {  // with so many of them on the chip
      const int latency = 92 + 8 * waves * ((workgroups + cus - 1) / cus), bandwidth = 47 * waves * workgroups / cus;
      return latency > bandwidth ? latency : bandwidth;
    };
    const int64_t full = step_time(slots);
    // (only the numbers of splits that shorten the longest one; none is empty then)
    for (int n = 1, per; n <= kTailMaxSplits && n <= most; n = (steps - 1) / (per - 1) + 1) {
      per = (steps + n - 1) / n;
      const int64_t total = wgs * n, rounds = total / slots;
      const int rest = (int)(total - rounds * slots);
      int64_t cost;
      if (once) {
        cost = rounds * (per * full + 224) + (rest ? (int64_t)per * step_time(rest) + 224 : 0);
        if (n > 1) cost += 227 + 47 * total * rows / (16 * cus);  // (the merge; the partial results out and in)
      } else {  // (bound by the products: whole rounds, each its steps and about one more)
        cost = (rounds + (rest > 0)) * (per + 1);
      }
      if (best < 0 || cost < best) {
        best = cost;
        t.waves = waves;
        t.nsplit = n;
        t.keys_per_split = per * unit;
      }
      if (per == 1) break;
    }
  }
  return t;
}

// The caller sizes part_o [B*nq*Hkv*rep*splits, D] fp32 and part_lse with it.
extern "C" int moba_tail_splits(int B, int Hkv, int rep, int nq, int Skv) {
  if (B <= 0 || Hkv <= 0 || rep <= 0 || nq <= 0 || nq > Skv || (int64_t)rep * nq > (1 << 20)) return 0;
  return tail_split(B, Hkv, rep * nq, Skv).nsplit;
}
extern "C" int moba_decode_splits(int B, int Hkv, int Skv) {
  return moba_tail_splits(B, Hkv, 1, 1, Skv);  // (the same for every group of up to 32 query heads)
}

template <class E>
static int launch_tail(const void* q, const void* k, const void* v, void* out, float* part_o, float* part_lse,
                       const TailSplit& ts, int B, int Hkv, int rep, int nq, int Skv, const int64_t* strides, float scale,
                       hipStream_t st) {
  LaunchCheck launch_check;
  typedef typename E::elem elem;
  TailParams<E> p;
  p.q = (const elem*)q; p.k = (const elem*)k; p.v = (const elem*)v; p.out = (elem*)out;
  p.part_o = part_o; p.part_lse = part_lse;
  p.q_stride_b = strides[0]; p.q_stride_h = strides[1]; p.q_stride_t = strides[2];
  p.kv_stride_b = strides[3]; p.kv_stride_h = strides[4];
  p.Hkv = Hkv; p.rep = rep; p.Skv = Skv; p.nq = nq;
  p.wr_log2 = ts.wr_log2; p.keys_per_split = ts.keys_per_split; p.nsplit = ts.nsplit;
  p.scale_log2 = scale * 1.4426950408889634f;
  static bool allowed[4][kMaxDevices];  // one set per element type
  typedef void (*Kernel)(TailParams<E>);
  static const Kernel kernels[4] = {tail_partial_kernel<E, false, 4>, tail_partial_kernel<E, true, 4>,
                                    tail_partial_kernel<E, true, 2>, tail_partial_kernel<E, true, 1>};
  const int form = ts.wr_log2 > 0 ? 0 : (ts.waves == 4 ? 1 : (ts.waves == 2 ? 2 : 3));
  const Kernel kernel = kernels[form];
  const int lds = ts.waves * kTailWaveLds;
  if (!allow_dynamic_lds((const void*)kernel, lds, allowed[form])) return MOBA_ERR_LAUNCH;
  hipLaunchKernelGGL(kernel, dim3(ts.nsplit, Hkv * ts.groups, B), dim3(64 * ts.waves), lds, st, p);
  if (ts.nsplit > 1)
    hipLaunchKernelGGL(tail_merge_kernel<E>, dim3((unsigned)((int64_t)B * nq * Hkv * rep)), dim3(256), 0, st,
                       (const float*)part_o, (const float*)part_lse, (elem*)out, ts.nsplit);
  return launch_check.result();
}

// q [B, H, nq, D] with the strides (elements) {batch, head, token}, D contiguous; k, v [B, Hkv, Skv, D] with the
// strides {batch, head}, a key row D contiguous elements and rows D apart: strides[5] holds the five.
// out [B, nq, H, D] contiguous.
extern "C" int moba_tail(const void* q, const void* k, const void* v, void* out, float* part_o, float* part_lse, int B,
                         int H, int Hkv, int nq, int Skv, int D, const int64_t* strides, float scale, int dtype,
                         void* stream) {
  if (!q || !k || !v || !out || !part_o || !part_lse || !strides) return MOBA_ERR_ARG;
  if (B <= 0 || H <= 0 || Hkv <= 0 || Skv <= 0 || nq <= 0 || nq > Skv || H % Hkv != 0 || B > 65535) return MOBA_ERR_ARG;
  if (D != kHeadDim || (dtype != MOBA_DTYPE_BF16 && dtype != MOBA_DTYPE_F16)) return MOBA_ERR_UNSUPPORTED;
  if (((uintptr_t)q & 15) || ((uintptr_t)k & 15) || ((uintptr_t)v & 15)) return MOBA_ERR_ARG;
  for (int i = 0; i < 5; ++i)
    if (strides[i] & 7) return MOBA_ERR_ARG;  // 16-byte loads
  const int rep = H / Hkv;
  if ((int64_t)rep * nq > (1 << 20)) return MOBA_ERR_LIMIT;
  const TailSplit ts = tail_split(B, Hkv, rep * nq, Skv);
  if ((int64_t)Hkv * ts.groups > 65535 || (int64_t)B * nq * H >= 0x7fffffffLL) return MOBA_ERR_LIMIT;
  hipStream_t st = (hipStream_t)stream;
  return dtype == MOBA_DTYPE_F16
             ? launch_tail<F16>(q, k, v, out, part_o, part_lse, ts, B, Hkv, rep, nq, Skv, strides, scale, st)
             : launch_tail<Bf16>(q, k, v, out, part_o, part_lse, ts, B, Hkv, rep, nq, Skv, strides, scale, st);
}

// One token: q [B, H, D] (strides q_stride_b, q_stride_h in elements), out [B, H, D] contiguous.  H / Hkv at most 32.
extern "C" int moba_decode(const void* q, const void* k, const void* v, void* out, float* part_o, float* part_lse,
                           int B, int H, int Hkv, int Skv, int D, int64_t q_stride_b, int64_t q_stride_h,
                           int64_t kv_stride_b, int64_t kv_stride_h, float scale, int dtype, void* stream) {
  if (Hkv > 0 && H / Hkv > 32) return MOBA_ERR_UNSUPPORTED;  // (moba_decode_splits knows groups of up to 32 only)
  const int64_t strides[5] = {q_stride_b, q_stride_h, 0, kv_stride_b, kv_stride_h};
  return moba_tail(q, k, v, out, part_o, part_lse, B, H, Hkv, 1, Skv, D, strides, scale, dtype, stream);
}
