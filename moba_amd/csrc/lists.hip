// Varlen gather lists: for every (filtered chunk f, head h) the ascending list of
// query tokens that selected it, as a counting sort keyed by (f, h) that is stable
// in the token index -- integer work, no copy of q or kv.
//
//   pass 1  count    one workgroup per (query chunk, head): how many of its tokens
//                    picked each earlier chunk of the sequence -> cnt[(f, h, query chunk)]
//   pass 2  scan     exclusive prefix sum (one workgroup, or two launches of many) of cnt in (f, h, query chunk) order: that is
//                    the list position of the first such token, because query chunks
//                    of a sequence are visited in ascending token order
//   pass 3  fill     same decomposition as pass 1; inside a workgroup the four waves own
//                    consecutive quarters of the chunk, and inside a 64-token batch
//                    the rank of a token among those with the same pick comes from a
//                    64-bit lane mask built with LDS atomics (order independent)
//   pass 4  segment offsets and per-segment tile counts, then their prefix sum
//
// List entries are destination rows of the partial-result buffers:
// dest = (token * H + h) * (K + 1) + 1 + slot, from which the token is recovered by
// one division.
#include "common.h"

namespace moba {

__device__ __forceinline__ int cnt_index(const int* __restrict__ pair_off, int f, int h, int H, int crel) {
  const int p0 = pair_off[f];
  const int nq = pair_off[f + 1] - p0;
  return p0 * H + h * nq + crel;
}

template <int NT>  // threads per workgroup
__global__ __launch_bounds__(NT) void lists_count_kernel(
    const int* __restrict__ sel, const int* __restrict__ chunk_tok, const int* __restrict__ chunk_fb,
    const int* __restrict__ chunk_local, const int* __restrict__ pair_off, int* __restrict__ cnt, int H, int K,
    int dense_local) {
  extern __shared__ int lds[];
  const int cq = blockIdx.x, h = blockIdx.y;
  const int c = chunk_local[cq];
  if (c == 0) return;
  const int fb = chunk_fb[cq];
  if (c <= dense_local) {  // a chunk of a dense prefix: its tokens have no list entries, its counts are zero
    for (int i = threadIdx.x; i < c; i += NT) cnt[cnt_index(pair_off, fb + i, h, H, c - i - 1)] = 0;
    return;
  }
  const int t0 = chunk_tok[cq], t1 = chunk_tok[cq + 1];
  for (int i = threadIdx.x; i < c; i += NT) lds[i] = 0;
  __syncthreads();
  for (int s = t0 + threadIdx.x; s < t1; s += NT) {
    const int* src = sel + ((int64_t)s * H + h) * K;
    for (int j = 0; j < K; ++j) {
      const int i = src[j] - fb;
      if ((unsigned)i < (unsigned)c) atomicAdd(&lds[i], 1);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < c; i += NT) cnt[cnt_index(pair_off, fb + i, h, H, c - i - 1)] = lds[i];
}

// the lanes of a wave see each other's LDS writes: a wave's LDS instructions execute in the order issued, so only
// the compiler has to be held to that order
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// KC: compile-time bound on K (a lane keeps its token's picks in registers); NW: waves of the workgroup, which
// own consecutive NW-ths of the chunk.  base_of() returns the scanned count array, in global memory or in LDS;
// it is called by the whole workgroup once the first loads of the picks are under way (it may synchronise).
template <int KC, int NW, class BaseFn>
__device__ __forceinline__ void lists_fill_body(
    const int* __restrict__ sel, const int* __restrict__ chunk_tok, const int* __restrict__ chunk_fb,
    const int* __restrict__ chunk_local, const int* __restrict__ pair_off, BaseFn base_of,
    int* __restrict__ seg_dest, int H, int K, int dense_local, int* lds) {
  const int cq = blockIdx.x, h = blockIdx.y;
  const int c_real = chunk_local[cq];
  const int c = c_real > dense_local ? c_real : 0;  // (no list entries from a chunk of a dense prefix)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int* pos = lds;                                             // [NW][c] running list position per wave
  unsigned* bits = reinterpret_cast<unsigned*>(lds + NW * c);  // [NW][c][2] lanes of the batch that picked i
  const int fb = chunk_fb[cq];
  const int t0 = chunk_tok[cq], t1 = chunk_tok[cq + 1];
  const int qlen = (t1 - t0 + NW - 1) / NW;
  const int w0 = min(t1, t0 + wave * qlen), w1 = min(t1, w0 + qlen);
  const int K1 = K + 1;
  // candidate index of each pick of this lane's token in a batch of 64, -1 when it is not a list entry
  auto load_picks = [&](int bi, int (&pick)[KC]) {
    const int s = w0 + bi * 64 + lane;
    const bool active = s < w1;
    const int* src = sel + ((int64_t)(active ? s : t0) * H + h) * K;
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      pick[j] = -1;
      if (j < K) {
        const int i = src[j] - fb;
        if (active && (unsigned)i < (unsigned)c) pick[j] = i;
      }
    }
  };
  constexpr int kKept = 2;  // the picks of the first batches stay in registers from the counting pass on
  int kept[kKept][KC];
#pragma unroll
  for (int bi = 0; bi < kKept; ++bi) load_picks(bi, kept[bi]);
  const int* base = base_of();
  if (c == 0) return;  // (the whole workgroup)
  for (int i = threadIdx.x; i < NW * c; i += NW * 64) {
    pos[i] = 0;
    bits[2 * i] = 0;
    bits[2 * i + 1] = 0;
  }
  __syncthreads();
  const int nbatch = (qlen + 63) / 64;  // same for all waves
  // per-wave counts
  for (int bi = 0; bi < nbatch; ++bi) {
    int pick[KC];
    if (bi < kKept) {
#pragma unroll
      for (int j = 0; j < KC; ++j) pick[j] = bi == 0 ? kept[0][j] : kept[1][j];
    } else {
      load_picks(bi, pick);
    }
#pragma unroll
    for (int j = 0; j < KC; ++j)
      if (pick[j] >= 0) atomicAdd(&pos[wave * c + pick[j]], 1);
  }
  __syncthreads();
  // counts -> start positions: global base of (f, h, this query chunk) plus the earlier waves
  for (int i = threadIdx.x; i < c; i += NW * 64) {
    int run = base[cnt_index(pair_off, fb + i, h, H, c - i - 1)];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const int n = pos[w * c + i];
      pos[w * c + i] = run;
      run += n;
    }
  }
  __syncthreads();
  // from here on a wave works on its own positions and lane masks only
  int* wpos = pos + wave * c;
  unsigned* wbits = bits + 2 * wave * c;
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int bi = 0; bi < nbatch; ++bi) {
    const int s = w0 + bi * 64 + lane;
    int pick[KC];
    if (bi < kKept) {
#pragma unroll
      for (int j = 0; j < KC; ++j) pick[j] = bi == 0 ? kept[0][j] : kept[1][j];
    } else {
      load_picks(bi, pick);
    }
#pragma unroll
    for (int j = 0; j < KC; ++j)
      if (pick[j] >= 0) atomicOr(&wbits[2 * pick[j] + (lane >> 5)], 1u << (lane & 31));
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      if (pick[j] >= 0) {
        const int i = pick[j];
        const uint64_t m = (uint64_t)wbits[2 * i] | ((uint64_t)wbits[2 * i + 1] << 32);
        const int rank = __popcll(m & below);
        seg_dest[wpos[i] + rank] = (s * H + h) * K1 + 1 + j;
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      if (pick[j] >= 0) {
        const int i = pick[j];
        const uint64_t m = (uint64_t)wbits[2 * i] | ((uint64_t)wbits[2 * i + 1] << 32);
        if ((m & below) == 0) {  // the first lane of this pick closes the batch for it
          wpos[i] += __popcll(m);
          wbits[2 * i] = 0;
          wbits[2 * i + 1] = 0;
        }
      }
    }
    wave_lds_sync();
  }
}

// NW waves per (query chunk, head): 4, or 16 for long chunks -- a wave walks its share of the chunk in batches of
// 64 tokens with three LDS round trips each, so the kernel's time is the number of batches per wave times that
// latency unless many waves are resident to hide it
template <int KC, int NW>
__global__ __launch_bounds__(NW * 64) void lists_fill_kernel(
    const int* __restrict__ sel, const int* __restrict__ chunk_tok, const int* __restrict__ chunk_fb,
    const int* __restrict__ chunk_local, const int* __restrict__ pair_off, const int* __restrict__ base,
    int* __restrict__ seg_dest, int H, int K, int dense_local) {
  extern __shared__ int lds[];
  lists_fill_body<KC, NW>(sel, chunk_tok, chunk_fb, chunk_local, pair_off, [&] { return base; }, seg_dest, H, K,
                          dense_local, lds);
}

// exclusive prefix sum of a[lo..hi) in place, starting from `carry`, by a workgroup of 1024; returns the total
__device__ __forceinline__ int scan_range(int* __restrict__ a, int lo, int hi, int carry) {
  __shared__ int wsum[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int half = 0;  // (two sets of wave sums in turn: one barrier per 4096 elements)
  for (int base = lo; base < hi; base += 4096, half ^= 1) {
    const int i0 = base + tid * 4;
    int v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (i0 + e < hi) ? a[i0 + e] : 0;
    const int tsum = v[0] + v[1] + v[2] + v[3];
    int inc = tsum;  // inclusive scan across the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[half][wave] = inc;
    __syncthreads();
    int woff = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int x = wsum[half][w];
      if (w < wave) woff += x;
      total += x;
    }
    int run = carry + woff + inc - tsum;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (i0 + e < hi) a[i0 + e] = run;
      run += v[e];
    }
    carry += total;
  }
  return carry;
}

// exclusive prefix sum of a[0..n) in place, total stored at a[n]; one workgroup.
__global__ __launch_bounds__(1024) void scan_kernel(int* __restrict__ a, int n) {
  const int total = scan_range(a, 0, n, 0);
  if (threadIdx.x == 0) a[n] = total;
}

// The same by many workgroups of `per` elements each, in two launches: the sums of the ranges, then every workgroup adds
// up the sums before its own and scans its range.  One workgroup alone is bound by its own round trips (4096 elements
// in about 2.5 us): 9.4 million counts -- 196608 tokens, 32 heads, chunks of 256 -- took it 5.8 ms of a call of 14 ms.
__global__ __launch_bounds__(1024) void scan_sums_kernel(const int* __restrict__ a, int n, int per, int* __restrict__ sums) {
  __shared__ int wsum[16];
  const int lo = blockIdx.x * per, hi = lo + min(n - lo, per);
  int s = 0;
  for (int i = lo + threadIdx.x; i < hi; i += 1024) s += a[i];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) s += wsum[w];
    sums[blockIdx.x] = s;
  }
}
__global__ __launch_bounds__(1024) void scan_apply_kernel(int* __restrict__ a, int n, int per, const int* __restrict__ sums) {
  __shared__ int wsum[16];
  int s = 0;
  for (int i = threadIdx.x; i < (int)blockIdx.x; i += 1024) s += sums[i];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s;
  __syncthreads();
  int carry = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) carry += wsum[w];
  const int lo = blockIdx.x * per, hi = lo + min(n - lo, per);
  const int total = scan_range(a, lo, hi, carry);
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) a[n] = total;
}

// List of (f, heads h .. h + n - 1) from the scanned counts: start and length.
__device__ __forceinline__ int2 list_range(const int* base, const int* __restrict__ pair_off, int fh, int H, int n) {
  const int f = fh / H, h = fh - f * H;
  const int p0 = pair_off[f], nq = pair_off[f + 1] - p0;
  const int start = base[p0 * H + h * nq];
  return make_int2(start, base[p0 * H + (h + n) * nq] - start);
}

// per (f, h): list start; per segment, the lists of G heads (1, or those of a key/value head): number of row tiles
__global__ __launch_bounds__(256) void lists_segments_kernel(const int* __restrict__ base,
                                                             const int* __restrict__ pair_off,
                                                             int* __restrict__ seg_off, int* __restrict__ tile_off,
                                                             int F, int H, int G, int tile_rows) {
  const int fh = blockIdx.x * 256 + threadIdx.x;
  if (fh > F * H) return;
  if (fh == F * H) {
    seg_off[fh] = base[pair_off[F] * H];
    return;
  }
  const int2 list = list_range(base, pair_off, fh, H, fh % G == 0 ? G : 1);
  seg_off[fh] = list.x;
  if (fh % G == 0) tile_off[fh / G] = (list.y + tile_rows - 1) / tile_rows;
}

// number of row tiles per segment of G heads from the list starts
__global__ __launch_bounds__(256) void lists_tile_counts_kernel(const int* __restrict__ seg_off,
                                                                int* __restrict__ tile_off, int segments, int G, int tile_rows) {
  const int s = blockIdx.x * 256 + threadIdx.x;
  if (s < segments) tile_off[s] = (seg_off[(s + 1) * G] - seg_off[s * G] + tile_rows - 1) / tile_rows;
}

// segment of every history tile id below `bound` (-1 past the last tile): the attention
// kernels then find their tile with one load instead of a search in tile_off
__global__ __launch_bounds__(256) void lists_tile_seg_kernel(const int* __restrict__ tile_off,
                                                             int* __restrict__ tile_seg, int FH, int bound) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= bound) return;
  tile_seg[t] = t < tile_off[FH] ? upper_row(tile_off, FH, t) : -1;
}

// Few segments and few tiles: what lists_segments_kernel (or lists_tile_counts_kernel, when `base` is null and
// seg_off is given), the scan of the tile counts and lists_tile_seg_kernel do, in one workgroup with the counts
// in LDS -- three dependent launches of a few microseconds each are most of the list stage of a small problem.
constexpr int kTailMaxSegments = 4096, kTailMaxTiles = 16384;
__global__ __launch_bounds__(1024) void lists_tail_kernel(const int* __restrict__ base, const int* __restrict__ pair_off,
                                                          int* __restrict__ seg_off, int* __restrict__ tile_off,
                                                          int* __restrict__ tile_seg, int F, int H, int G, int tile_rows,
                                                          int bound) {
  __shared__ int off[kTailMaxSegments + 1];
  __shared__ int wsum[16];
  const int FH = F * H / G, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;  // (FH: segments)
  if (base) {  // the list starts
    for (int fh = tid; fh <= F * H; fh += 1024)
      seg_off[fh] = fh == F * H ? base[pair_off[F] * H] : list_range(base, pair_off, fh, H, 1).x;
  }
  // this thread's four consecutive segments: tile counts
  int v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int s = tid * 4 + e;
    v[e] = 0;
    if (s < FH) v[e] = ((base ? list_range(base, pair_off, s * G, H, G).y : seg_off[(s + 1) * G] - seg_off[s * G]) + tile_rows - 1) / tile_rows;
  }
  const int tsum = v[0] + v[1] + v[2] + v[3];
  int inc = tsum;  // inclusive scan across the wave, then across the waves
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int woff = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const int x = wsum[w];
    if (w < wave) woff += x;
    total += x;
  }
  int run = woff + inc - tsum;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int fh = tid * 4 + e;
    if (fh < FH) {
      off[fh] = run;
      tile_off[fh] = run;
    }
    run += v[e];
  }
  if (tid == 0) {
    off[FH] = total;
    tile_off[FH] = total;
  }
  __syncthreads();
  for (int t = tid; t < bound; t += 1024) {
    int seg = -1;
    if (t < total) {
      int lo = 0, hi = FH;  // off[lo] <= t < off[hi]
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= t) lo = mid; else hi = mid;
      }
      seg = lo;
    }
    tile_seg[t] = seg;
  }
}

// Small problems: the scan, the fill and the tables in one launch.  Every workgroup scans the whole count array for itself
// into LDS (cheaper than a launch that does it once); workgroups (cq < N, h) fill their part of the lists, workgroups
// (N, h) write an H-th of the tables each, which depend on the scanned counts only.
// NW waves as in lists_fill_kernel: 16 for long chunks, 4 otherwise -- workgroups of 16 waves start one after the other, 22 ns
// apart, and a chunk of 512 tokens is half a batch for each.  Measured: 8191 tokens, 32 heads, chunk 512 (16 waves each
// and one of them for all tables before): 19.0 -> 15.9 us; 3 x 2001 tokens, 32 heads, chunk 256 (scan, fill and tables as
// three launches before): 17.3 -> 10.4 us; 20480 tokens, 8 heads, chunk 512: 11.8 -> 9.0; 4096 tokens, 4 heads, chunk
// 512: 6.4 -> 5.6.  The form of 16 waves is as fast as its forerunner, within 0.3 us, but for 256 workgroups and about 4000
// counts (32 chunks of 1024 tokens, 8 heads): 9.4 -> 10.5 us.
constexpr int kFusedMaxCounts = 8192, kFusedMaxCand = 128;
constexpr int64_t kFusedMaxWork = 1 << 22;
template <int KC, int NW>
__global__ __launch_bounds__(NW * 64) void lists_fill_tail_kernel(
    const int* __restrict__ sel, const int* __restrict__ chunk_tok, const int* __restrict__ chunk_fb,
    const int* __restrict__ chunk_local, const int* __restrict__ pair_off, const int* __restrict__ cnt,
    int* __restrict__ seg_dest, int* __restrict__ seg_off, int* __restrict__ tile_off, int* __restrict__ tile_seg,
    int N, int H, int K, int F, int PH, int G, int tile_rows, int bound, int Gb, int tile_rows_b,
    int* __restrict__ tile_off_b, int* __restrict__ tile_seg_b, int bound_b, int dense_local) {
  constexpr int NT = NW * 64, kSteps = kFusedMaxCounts / (4 * NT);
  // the scanned counts [PH + 1]; the tables' tile starts [F*H + 1], or the fill's positions and lane masks: NW x 3 ints per
  // candidate chunk
  extern __shared__ int lds[];
  __shared__ int wsum[kSteps][NW];
  int* const sbase = lds;
  int* const off = lds + PH + 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // inclusive sum over the workgroup's lanes up to this one within its wave
  auto wave_scan = [&](int x) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(x, o, 64);
      if (lane >= o) x += t;
    }
    return x;
  };
  // (asked for ahead of everything else: the fill's lookups and picks travel meanwhile)
  int v[kSteps][4];
#pragma unroll
  for (int st = 0; st < kSteps; ++st) {
    if (st * NT * 4 >= PH) break;  // (uniform; without it the loads of the empty steps, which return nothing, cost
                                   // 0.8 us of 6.4 at 8 chunks of 512, 4 heads, and 0.2 of 9.0 in the form of 16 waves)
    const int i0 = (st * NT + tid) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[st][e] = i0 + e < PH ? cnt[i0 + e] : 0;
  }
  auto scanned_counts = [&]() -> const int* {
    int inc[kSteps], sum[kSteps];
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      if (st * NT * 4 >= PH) break;  // (uniform)
      sum[st] = v[st][0] + v[st][1] + v[st][2] + v[st][3];
      inc[st] = wave_scan(sum[st]);
      if (lane == 63) wsum[st][wave] = inc[st];
    }
    __syncthreads();
    int carry = 0;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      if (st * NT * 4 >= PH) break;
      int woff = 0, total = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const int x = wsum[st][w];
        if (w < wave) woff += x;
        total += x;
      }
      int run = carry + woff + inc[st] - sum[st];
      const int i0 = (st * NT + tid) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (i0 + e < PH) sbase[i0 + e] = run;
        run += v[st][e];
      }
      carry += total;
    }
    if (tid == 0) sbase[PH] = carry;
    __syncthreads();
    return sbase;
  };
  if (blockIdx.x < N) {
    lists_fill_body<KC, NW>(sel, chunk_tok, chunk_fb, chunk_local, pair_off, scanned_counts, seg_dest, H, K, dense_local, off);
    return;
  }
  // the tables: this workgroup's share of the segments and of the tiles
  const int part = blockIdx.y;
  const int* base = scanned_counts();
  for (int fh = part * NT + tid; fh <= F * H; fh += H * NT)
    seg_off[fh] = fh == F * H ? base[PH] : list_range(base, pair_off, fh, H, 1).x;
  auto tables = [&](int G, int rows, int* toff, int* tseg, int nbound) {
    const int segments = F * H / G;
    int carry = 0;
    for (int s0 = 0; s0 < segments; s0 += NT) {
      const int s = s0 + tid;
      const int n = s < segments ? (list_range(base, pair_off, s * G, H, G).y + rows - 1) / rows : 0;
      const int inc = wave_scan(n);
      if (lane == 63) wsum[0][wave] = inc;
      __syncthreads();
      int woff = 0, total = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const int x = wsum[0][w];
        if (w < wave) woff += x;
        total += x;
      }
      const int at = carry + woff + inc - n;
      if (s < segments) {
        off[s] = at;
        if (s % H == part) toff[s] = at;
      }
      carry += total;
      __syncthreads();  // (the sums are read)
    }
    if (tid == 0) {
      off[segments] = carry;
      if (part == 0) toff[segments] = carry;
    }
    __syncthreads();
    const int t1 = (int)((int64_t)nbound * (part + 1) / H);
    for (int t = (int)((int64_t)nbound * part / H) + tid; t < t1; t += NT) {
      int seg = -1;
      if (t < carry) {
        int lo = 0, hi = segments;  // off[lo] <= t < off[hi]
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (off[mid] <= t) lo = mid; else hi = mid;
        }
        seg = lo;
      }
      tseg[t] = seg;
    }
  };
  tables(G, tile_rows, tile_off, tile_seg, bound);
  if (tile_off_b) {  // the same lists cut into tiles of another height (the backward kernels')
    __syncthreads();
    tables(Gb, tile_rows_b, tile_off_b, tile_seg_b, bound_b);
  }
}

}  // namespace moba

using namespace moba;

// scratch: scratch_ints ints that nobody needs until the scan is done.  Up to 16384 elements (four of its steps) one
// workgroup costs no more than the second launch.
static void launch_scan(int* a, int n, int* scratch, int64_t scratch_ints, hipStream_t st) {
  int64_t groups = ((int64_t)n + 4095) / 4096;
  if (groups > scratch_ints) groups = scratch_ints;
  if (n <= 16384 || groups < 2) {
    hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(1024), 0, st, a, n);
    return;
  }
  const int64_t steps = ((int64_t)n + groups * 4096 - 1) / (groups * 4096);  // per workgroup
  const int per = (int)(steps * 4096);
  const dim3 grid((unsigned)(((int64_t)n + per - 1) / per));
  hipLaunchKernelGGL(scan_sums_kernel, grid, dim3(1024), 0, st, (const int*)a, n, per, scratch);
  hipLaunchKernelGGL(scan_apply_kernel, grid, dim3(1024), 0, st, a, n, per, (const int*)scratch);
}

static void launch_tile_tables(const int32_t* seg_off, int32_t* tile_off, int32_t* tile_seg, int H, int F, int G,
                               int tile_rows, int64_t hist_bound, hipStream_t st) {
  const int segments = F * H / G;
  if (segments < kTailMaxSegments && hist_bound <= kTailMaxTiles) {
    hipLaunchKernelGGL(lists_tail_kernel, dim3(1), dim3(1024), 0, st, (const int*)nullptr, (const int*)nullptr,
                       const_cast<int*>(seg_off), tile_off, tile_seg, F, H, G, tile_rows, (int)hist_bound);
    return;
  }
  hipLaunchKernelGGL(lists_tile_counts_kernel, dim3((segments + 255) / 256), dim3(256), 0, st, seg_off, tile_off, segments, G,
                     tile_rows);
  launch_scan(tile_off, segments, tile_seg, hist_bound, st);
  hipLaunchKernelGGL(lists_tile_seg_kernel, dim3((unsigned)((hist_bound + 255) / 256)), dim3(256), 0, st,
                     (const int*)tile_off, tile_seg, segments, (int)hist_bound);
}

// Limits: chunks per sequence minus one (cmax) is bounded by the LDS the fill pass
// needs, 12 bytes per wave and candidate chunk (4 waves up to 3413 chunks, one wave up to 13653).
extern "C" int moba_build_lists_grouped(const int32_t* sel, const int32_t* chunk_tok, const int32_t* chunk_fb,
                                const int32_t* chunk_local, const int32_t* pair_off, int32_t* cnt,
                                int32_t* seg_off, int32_t* tile_off, int32_t* seg_dest, int32_t* tile_seg,
                                int64_t S, int H, int K, int N, int F, int P, int cmax, int tile_rows,
                                int64_t hist_bound, int counted, int tile_rows_b, int32_t* tile_off_b,
                                int32_t* tile_seg_b, int64_t hist_bound_b, int dense_local, int list_heads,
                                int list_heads_b, void* stream) {
  LaunchCheck launch_check;
  if (!sel || !chunk_tok || !chunk_fb || !chunk_local || !pair_off || !cnt || !seg_off || !tile_off || !seg_dest ||
      !tile_seg)
    return MOBA_ERR_ARG;
  if (hist_bound <= 0 || hist_bound >= 0x7fffffffLL) return MOBA_ERR_ARG;
  if (tile_off_b && (!tile_seg_b || tile_rows_b <= 0 || hist_bound_b <= 0 || hist_bound_b >= 0x7fffffffLL))
    return MOBA_ERR_ARG;
  if (S <= 0 || H <= 0 || K <= 0 || N <= 0 || F <= 0 || P <= 0 || cmax <= 0 || tile_rows <= 0) return MOBA_ERR_ARG;
  if (dense_local < 0 || dense_local > K) return MOBA_ERR_ARG;
  if (list_heads <= 0 || H % list_heads != 0 || list_heads_b <= 0 || H % list_heads_b != 0) return MOBA_ERR_ARG;
  if ((int64_t)S * H * (K + 1) >= 0x7fffffffLL || (int64_t)P * H > 0x7fffffffLL - 4096) return MOBA_ERR_LIMIT;
  // (the scan's steps of 4096 counts stay within an int)
  if (H > 65535 || (size_t)cmax * 12 > 160 * 1024) return MOBA_ERR_LIMIT;
  hipStream_t st = (hipStream_t)stream;
  dim3 grid(N, H);
  const bool small_tail = (int64_t)F * H < kTailMaxSegments && hist_bound <= kTailMaxTiles;
  // One launch for all: its workgroups scan all counts each, so it is for few counts times workgroups; of 16 waves where a
  // chunk's batches of 64 tokens are many for four, the workgroups few.  A chunk's length is not known here but between
  // S / N and S / F, as only the last chunk of a sequence is shorter: with that one half as long it is 2 S / (N + F).
  // (The line by S / N >= 1024 missed most sequences that end within a chunk of 1024.)  4 waves / 16 waves in us, up to 64
  // workgroups: 1 to 4 picks: chunk 512: 5.7 / 6.3; 768: 7.1 / 6.9; 1024: 8.6 / 7.5; 7 and 11 picks: 320: 10.5 / 9.9;
  // 512: 10.5 / 10.5; 640: 15.0 / 11.4.  256 workgroups: 1 to 4 picks: 768:
  // 9.7 / 10.2; 896: 11.6 / 11.0; 7 and 11 picks: 512: 16.7 / 18.0; 640: 22.4 / 20.4.  512 workgroups, 2 picks: 1024:
  // 15.7 / 17.9; 2048: 27.2 / 26.0.
  const int64_t counts = (int64_t)P * H, groups = (int64_t)N * H, rows = 2 * S / ((int64_t)N + F);
  const bool many_waves = rows >= (K > 4 ? 576 : 704) ? groups <= (rows >= 1024 ? 512 : 256)
                                                      : K > 4 && rows >= 288 && groups <= 64;
  if (small_tail && counts <= kFusedMaxCounts && cmax <= kFusedMaxCand && groups * counts <= kFusedMaxWork && K <= 16 &&
      (!tile_off_b || hist_bound_b <= kTailMaxTiles)) {
    if (!counted)
      hipLaunchKernelGGL(lists_count_kernel<256>, grid, dim3(256), (size_t)cmax * 4, st, sel, chunk_tok, chunk_fb,
                         chunk_local, pair_off, cnt, H, K, dense_local);
    const int nw = many_waves ? 16 : 4, tables = F * H + 1, fill = nw * 3 * cmax;
    const size_t lds = ((size_t)counts + 1 + (tables > fill ? tables : fill)) * 4;  // (at most 56 KiB)
#define MOBA_FILL_TAIL(KC, NW)                                                                                       \
  hipLaunchKernelGGL((lists_fill_tail_kernel<KC, NW>), dim3(N + 1, H), dim3(NW * 64), lds, st, sel, chunk_tok, chunk_fb, \
                     chunk_local, pair_off, (const int*)cnt, seg_dest, seg_off, tile_off, tile_seg, N, H, K, F,      \
                     P * H, list_heads, tile_rows, (int)hist_bound, list_heads_b, tile_rows_b, tile_off_b, tile_seg_b, (int)hist_bound_b,      \
                     dense_local)
    if (K <= 4) {
      if (many_waves) MOBA_FILL_TAIL(4, 16); else MOBA_FILL_TAIL(4, 4);
    } else {
      if (many_waves) MOBA_FILL_TAIL(16, 16); else MOBA_FILL_TAIL(16, 4);
    }
#undef MOBA_FILL_TAIL
    return launch_check.result();
  }
  if (!counted)
    hipLaunchKernelGGL(lists_count_kernel<256>, grid, dim3(256), (size_t)cmax * 4, st, sel, chunk_tok, chunk_fb,
                       chunk_local, pair_off, cnt, H, K, dense_local);
  // (scratch: the list starts, F*H+1 ints that the launches behind the scan write.  The tile tables are shorter where heads
  // are cut together, and the sums -- one per 4096 counts -- can be more than they hold.)
  launch_scan(cnt, P * H, seg_off, (int64_t)F * H, st);
  // more than 64 KiB of dynamic LDS has to be asked for explicitly
  // (LDS: 12 bytes per wave and candidate chunk)
  const bool wide = S / N >= 1024 && (size_t)cmax * 192 <= 64 * 1024;  // long chunks: 16 waves per (chunk, head)
#define MOBA_FILL(KC)                                                                                          \
  {                                                                                                            \
    if (wide) {                                                                                                \
      hipLaunchKernelGGL((lists_fill_kernel<KC, 16>), grid, dim3(1024), (size_t)cmax * 192, st, sel, chunk_tok, \
                         chunk_fb, chunk_local, pair_off, (const int*)cnt, seg_dest, H, K, dense_local);       \
    } else if ((size_t)cmax * 48 <= 160 * 1024) {                                                              \
      if ((size_t)cmax * 48 > 64 * 1024 &&                                                                     \
          hipFuncSetAttribute((const void*)lists_fill_kernel<KC, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                              (int)((size_t)cmax * 48)) != hipSuccess)                                         \
        return MOBA_ERR_LAUNCH;                                                                                \
      hipLaunchKernelGGL((lists_fill_kernel<KC, 4>), grid, dim3(256), (size_t)cmax * 48, st, sel, chunk_tok,   \
                         chunk_fb, chunk_local, pair_off, (const int*)cnt, seg_dest, H, K, dense_local);       \
    } else { /* very many chunks per sequence: one wave, so that its tables still fit */                       \
      if (hipFuncSetAttribute((const void*)lists_fill_kernel<KC, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                              (int)((size_t)cmax * 12)) != hipSuccess)                                         \
        return MOBA_ERR_LAUNCH;                                                                                \
      hipLaunchKernelGGL((lists_fill_kernel<KC, 1>), grid, dim3(64), (size_t)cmax * 12, st, sel, chunk_tok,    \
                         chunk_fb, chunk_local, pair_off, (const int*)cnt, seg_dest, H, K, dense_local);       \
    }                                                                                                          \
  }
  if (K <= 4) MOBA_FILL(4)
  else if (K <= 16) MOBA_FILL(16)
  else if (K <= 64) MOBA_FILL(64)
  else return MOBA_ERR_LIMIT;
#undef MOBA_FILL
  if (small_tail) {
    hipLaunchKernelGGL(lists_tail_kernel, dim3(1), dim3(1024), 0, st, (const int*)cnt, pair_off, seg_off, tile_off,
                       tile_seg, F, H, list_heads, tile_rows, (int)hist_bound);
  } else {
    hipLaunchKernelGGL(lists_segments_kernel, dim3((F * H + 1 + 255) / 256), dim3(256), 0, st, (const int*)cnt,
                       pair_off, seg_off, tile_off, F, H, list_heads, tile_rows);
    launch_scan(tile_off, F * H / list_heads, tile_seg, hist_bound, st);
    hipLaunchKernelGGL(lists_tile_seg_kernel, dim3((unsigned)((hist_bound + 255) / 256)), dim3(256), 0, st,
                       (const int*)tile_off, tile_seg, F * H / list_heads, (int)hist_bound);
  }
  if (tile_off_b) launch_tile_tables(seg_off, tile_off_b, tile_seg_b, H, F, list_heads_b, tile_rows_b, hist_bound_b, st);
  return launch_check.result();
}

extern "C" int moba_build_lists(const int32_t* sel, const int32_t* chunk_tok, const int32_t* chunk_fb,
                                const int32_t* chunk_local, const int32_t* pair_off, int32_t* cnt,
                                int32_t* seg_off, int32_t* tile_off, int32_t* seg_dest, int32_t* tile_seg,
                                int64_t S, int H, int K, int N, int F, int P, int cmax, int tile_rows,
                                int64_t hist_bound, int counted, int tile_rows_b, int32_t* tile_off_b,
                                int32_t* tile_seg_b, int64_t hist_bound_b, int dense_local, void* stream) {
  return moba_build_lists_grouped(sel, chunk_tok, chunk_fb, chunk_local, pair_off, cnt, seg_off, tile_off, seg_dest, tile_seg,
                                  S, H, K, N, F, P, cmax, tile_rows, hist_bound, counted, tile_rows_b, tile_off_b, tile_seg_b,
                                  hist_bound_b, dense_local, 1, 1, stream);
}

// The tile tables alone, for another number of rows per tile, from the list starts moba_build_lists wrote
// (the forward and the backward kernels cut the same lists into tiles of different heights).
extern "C" int moba_tile_tables(const int32_t* seg_off, int32_t* tile_off, int32_t* tile_seg, int H, int F,
                                int tile_rows, int64_t hist_bound, void* stream) {
  LaunchCheck launch_check;
  if (!seg_off || !tile_off || !tile_seg) return MOBA_ERR_ARG;
  if (H <= 0 || F <= 0 || tile_rows <= 0 || hist_bound <= 0 || hist_bound >= 0x7fffffffLL) return MOBA_ERR_ARG;
  if ((int64_t)F * H >= 0x7fffffffLL) return MOBA_ERR_LIMIT;
  launch_tile_tables(seg_off, tile_off, tile_seg, H, F, 1, tile_rows, hist_bound, (hipStream_t)stream);
  return launch_check.result();
}
