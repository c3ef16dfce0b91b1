// Key chunk-mean: kbar[f, h, :] = round( mean over the B tokens of filtered chunk f of K[., h, :] ),
// rounded once to the element type (bf16 or fp16).
//
// HBM-bound: K is read exactly once with 16-byte loads (a wave covers 1 KiB of
// one token row); the algorithmic traffic is S*H*D*2 bytes.  Accumulation is
// in fp64: the sum of a chunk of 16-bit float values is then exact, so the result
// does not depend on how the chunk is split over workgroups, and the rounded
// mean is reproducible bit for bit (fp64 -> fp32 -> element type, round to nearest even).
//
// One stage (chunk_mean_whole_kernel): one workgroup of 256 to 1024 threads per (chunk, head) or part of its columns
//          (column_parts_log2), column groups of 8 times the token lanes, their sums added through LDS: one launch instead of
//          two, and no partial sums in memory.  131072 tokens, 8 heads, chunk 4096: 67 -> 44 us; 302060 tokens, 32 heads,
//          chunk 2048: 474 -> 389 us; in halves, 32768 tokens, one head, chunk 1024: 10.2 -> 9.2 us (keys just written).
// Two stages for very many short chunks, and where one would leave few workgroups for very many bytes each (see whole_chunks):
//   Stage 1: grid (F, token splits, column blocks); each thread owns 8 adjacent
//            columns of the [H*D] token row and sums its share of a token split.
//   Stage 2: sums the splits in order, divides by B, rounds.
#include <mutex>
#include "common.h"

namespace moba {

// cpb_log2: the workgroup's 256 threads are 1 << cpb_log2 column groups (8 adjacent columns each) times
// 256 >> cpb_log2 token lanes: a row narrower than 2048 elements still occupies every lane, and the token lanes'
// sums are added through LDS (exact sums: the order does not matter).
template <class E>
__global__ __launch_bounds__(256) void chunk_mean_partial_kernel(
    const typename E::elem* __restrict__ k, const int* __restrict__ fchunk_tok, double* __restrict__ partial,
    int HD8 /* H*D/8 */, int D8 /* D/8 */, int B, int nsplit, int tok_per_split, int64_t row_stride,
    int64_t head_stride, int batch_rows, int64_t batch_stride, int cpb_log2, int* __restrict__ clear,
    int64_t clear_ints) {
  MOBA_ELEM_TYPES(E)
  __shared__ double red[256 * 8];
  if (clear) {  // an int array of the caller's to be zeroed on the way (the workgroups share it out)
    const int64_t wg = blockIdx.x + (int64_t)gridDim.x * (blockIdx.y + (int64_t)gridDim.y * blockIdx.z);
    const int64_t step = (int64_t)gridDim.x * gridDim.y * gridDim.z * 256;
    for (int64_t i = wg * 256 + threadIdx.x; i < clear_ints; i += step) clear[i] = 0;
  }
  const int cpb = 1 << cpb_log2, lanes = 256 >> cpb_log2;
  const int tl = threadIdx.x >> cpb_log2;
  const int col = blockIdx.z * cpb + (threadIdx.x & (cpb - 1));
  const bool col_ok = col < HD8;
  const int split = blockIdx.y;
  const int f = blockIdx.x;  // the only grid dimension without a 65535 limit
  const int t0 = split * tok_per_split;
  const int t1 = min(B, t0 + tok_per_split);
  const int head = col_ok ? col / D8 : 0;
  // (a chunk lies inside one sequence, hence inside one batch entry of a batched layout)
  const int tok0 = fchunk_tok[f];
  const int be = batch_rows ? tok0 / batch_rows : 0;
  const elem* src = k + be * batch_stride + ((int64_t)(tok0 - be * batch_rows) + t0 + tl) * row_stride +
                    head * head_stride + (col_ok ? col - head * D8 : 0) * 8;
  const int64_t step = (int64_t)lanes * row_stride;
  double acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0;
  int t = t0 + tl;
  if (col_ok) {
    for (; t + 7 * lanes < t1; t += 8 * lanes) {
      elem8 x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = __builtin_nontemporal_load(reinterpret_cast<const elem8*>(src + u * step));
      src += 8 * step;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        // sums of 16-bit float values are exact in fp64 whatever the order
        const double a = ((double)(float)x[0][e] + (double)(float)x[1][e]) + ((double)(float)x[2][e] + (double)(float)x[3][e]);
        const double b = ((double)(float)x[4][e] + (double)(float)x[5][e]) + ((double)(float)x[6][e] + (double)(float)x[7][e]);
        acc[e] += a + b;
      }
    }
    for (; t < t1; t += lanes) {
      elem8 x0 = *reinterpret_cast<const elem8*>(src);
      src += step;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += (double)(float)x0[e];
    }
  }
  if (lanes > 1) {  // (uniform)
#pragma unroll
    for (int e = 0; e < 8; ++e) red[e * 256 + threadIdx.x] = acc[e];
    __syncthreads();
    if (tl != 0) return;
    for (int l = 1; l < lanes; ++l)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += red[e * 256 + (l << cpb_log2) + threadIdx.x];
  }
  if (!col_ok) return;
  double* dst = partial + ((int64_t)(f * nsplit + split) * HD8 + col) * 8;
#pragma unroll
  for (int e = 0; e < 8; ++e) dst[e] = acc[e];
}

// fp64 -> fp32 rounded to odd (an inexact result gets the neighbour whose last bit is set): rounding that fp32
// value to bf16 or fp16 to nearest-even then gives what rounding the fp64 value once would, where two
// nearest-even roundings in a row can land on the wrong side of a tie.
__device__ __forceinline__ float round_to_odd_f32(double x) {
  float f = (float)x;  // nearest-even
  if ((double)f != x) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if (fabs((double)f) > fabs(x)) u -= 1;  // the neighbour toward zero (never crosses zero: |f| > |x| >= 0)
    u |= 1;
    f = __builtin_bit_cast(float, u);
  }
  return f;
}

// One workgroup of NT threads per (chunk f, head, part of the columns): thread (tl, c) sums the tokens tl, tl + lanes, ... of
// the part's columns 8c .. 8c + 7.  D8 column groups, a power of two up to 16.  NT: about eight tokens per lane or more, so that every
// lane has its eight rows in flight and the sums' way through LDS stays short against them (65536 tokens, 8 heads, chunk
// 128: 53 us with 1024 threads, 22 with 256).
template <class E, int NT>
__global__ __launch_bounds__(NT) void chunk_mean_whole_kernel(
    const typename E::elem* __restrict__ k, const int* __restrict__ fchunk_tok, typename E::elem* __restrict__ kbar,
    int d8_log2, int B, int64_t row_stride, int64_t head_stride, int batch_rows, int64_t batch_stride,
    int* __restrict__ clear, int64_t clear_ints) {  // d8_log2: of the column groups of this workgroup's part
  MOBA_ELEM_TYPES(E)
  __shared__ double red[8][NT / 64][16];  // [element][wave][column group]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int f = blockIdx.x, head = blockIdx.y, H = gridDim.y, part = blockIdx.z;
  if (clear) {
    const int64_t step = (int64_t)gridDim.x * H * gridDim.z * NT;
    for (int64_t i = (((int64_t)part * H + head) * gridDim.x + f) * NT + tid; i < clear_ints; i += step) clear[i] = 0;
  }
  const int D8 = 1 << d8_log2, lanes = NT >> d8_log2;
  const int c = tid & (D8 - 1), tl = tid >> d8_log2;
  const int col0 = part * D8 * 8, D = gridDim.z * D8 * 8;
  const int tok0 = fchunk_tok[f];
  const int be = batch_rows ? tok0 / batch_rows : 0;  // (a chunk lies inside one batch entry)
  const elem* src = k + be * batch_stride + ((int64_t)(tok0 - be * batch_rows) + tl) * row_stride + head * head_stride + col0 + c * 8;
  const int64_t step = (int64_t)lanes * row_stride;
  double acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0;
  int t = tl;
  for (; t + 7 * lanes < B; t += 8 * lanes) {
    elem8 x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = __builtin_nontemporal_load(reinterpret_cast<const elem8*>(src + u * step));
    src += 8 * step;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const double a = ((double)(float)x[0][e] + (double)(float)x[1][e]) + ((double)(float)x[2][e] + (double)(float)x[3][e]);
      const double b = ((double)(float)x[4][e] + (double)(float)x[5][e]) + ((double)(float)x[6][e] + (double)(float)x[7][e]);
      acc[e] += a + b;
    }
  }
  {  // the rest (up to seven rows), requested together
    elem8 x[7];
#pragma unroll
    for (int u = 0; u < 7; ++u)
      if (t + u * lanes < B) x[u] = __builtin_nontemporal_load(reinterpret_cast<const elem8*>(src + u * step));
#pragma unroll
    for (int u = 0; u < 7; ++u)
      if (t + u * lanes < B)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += (double)(float)x[u][e];
  }
  // the token lanes of a wave, then the waves (exact sums: the order does not matter)
  for (int o = D8; o < 64; o <<= 1)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], o, 64);
  if (lane < D8)
#pragma unroll
    for (int e = 0; e < 8; ++e) red[e][wave][lane] = acc[e];
  __syncthreads();
  if (tid >= 8 * D8) return;
  const int e = tid >> d8_log2;  // element e of column group c
  double sum = 0.0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) sum += red[e][w][c];
  kbar[((int64_t)f * H + head) * D + col0 + c * 8 + e] = (elem)round_to_odd_f32(sum / (double)B);
}

template <class E>
__global__ __launch_bounds__(64) void chunk_mean_finish_kernel(
    const double* __restrict__ partial, typename E::elem* __restrict__ kbar, int HD8, int B, int nsplit, int F) {
  MOBA_ELEM_TYPES(E)
  // (one wave per workgroup: a small problem's few hundred outputs then spread over several compute units)
  const int64_t idx = (int64_t)blockIdx.x * 64 + threadIdx.x;  // over F * HD8
  if (idx >= (int64_t)F * HD8) return;
  const int f = (int)(idx / HD8);
  const int col = (int)(idx % HD8);
  double acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0;
  const double* src = partial + ((int64_t)f * nsplit * HD8 + col) * 8;
  const int64_t step = (int64_t)HD8 * 8;
  int s = 0;
  for (; s + 4 <= nsplit; s += 4) {  // four splits' loads in flight together (nsplit is a power of two)
    double x[4][8];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[u][e] = src[u * step + e];
    src += 4 * step;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += (x[0][e] + x[1][e]) + (x[2][e] + x[3][e]);
  }
  for (; s < nsplit; ++s, src += step)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += src[e];
  elem8 o;
  const double inv = (double)B;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (elem)round_to_odd_f32(acc[e] / inv);
  *reinterpret_cast<elem8*>(kbar + idx * 8) = o;
}

}  // namespace moba

using namespace moba;

// column groups per workgroup (as a power of two): all 256 threads for rows of 2048 elements or more
static int pick_cpb_log2(int HD8) {
  int c = 0;
  while (c < 8 && (1 << c) < HD8) ++c;
  return c;
}
static int pick_nsplit(int HD8, int F, int B) {
  const int cpb_log2 = pick_cpb_log2(HD8);
  const int colblocks = (HD8 + (1 << cpb_log2) - 1) >> cpb_log2;
  const int lanes = 256 >> cpb_log2;
  int nsplit = 1;
  // enough workgroups to keep every CU's memory pipeline full (8 row loads in flight per lane),
  // few enough that the fp64 partial sums stay a small fraction of the traffic
  while ((int64_t)colblocks * F * nsplit < 1536 && B / (nsplit * 2) >= 64 && B / (nsplit * 2) >= 8 * lanes) nsplit *= 2;
  return nsplit;
}

extern "C" size_t moba_chunk_mean_workspace_bytes(int H, int D, int F, int B) {
  if (H <= 0 || D <= 0 || F <= 0 || B <= 0 || (H * D) % 8 != 0) return 0;
  const int HD8 = H * D / 8;
  return (size_t)F * pick_nsplit(HD8, F, B) * HD8 * 8 * sizeof(double);
}

// Times below: us with the keys last written before 640 MB of other data / just before the call; two stages with both launches.
//
// Into how many parts (log2) the columns of a chunk and head go, each a workgroup's.  Halves of 128-element heads below 128
// (chunk, head) pairs: whole rows leave compute units without a workgroup there, and a workgroup's reads are a chain of its own
// length; from there on they only make a second round.  Parts of 64 bytes, half a line of the caches, only for up to 64 pairs
// and 17 MB, and only where the two workgroups of a line share a second-level cache: workgroups go to the eight XCDs in turn
// and a part's numbers lie F * H behind those of the part before, so where 8 divides that; elsewhere each line is fetched twice.
// Whole rows / halves / quarters, 128-element heads (heads x chunks, tokens a chunk): 1 x 15, 2048: 17.3 / 14.3, 12.8 / 10.4, 12.8 /
// 13.0; 1 x 31, 1024: 12.1 / 10.2, 10.4 / 9.2, 10.2 / 10.4; 8 x 1, 4096: 29.1 / 22.2, 21.1 / 14.8, 18.6 / 13.3; 8 x 3, 2048: -, 14.4 /
// 11.2, 13.7 / 11.1; 8 x 7, 4096: 31.9 / 23.5, 23.7 / 18.6, 21.9 / 27.2; 8 x 15, 1024: 14.1 / 12.8, 12.8 / 12.9, 13.6 / 15.1; 4 x 31,
// 4096: 35.2 / 35.6, 31.2 / 42.0, 51 / 62; 32 x 5, 1024: 14.6 / 14.2, 19.0 / 18.1, 18.2 / 21.9; 1 x 190, 1024: 15.3 / 15.3, 18.9 / 19.6,
// 22.9 / 25.6; 64-element heads, whole rows / halves: 8 x 1, 4096: 21.4 / 14.8, 19.0 / 13.3; 8 x 7, 1024: 10.8 / 9.2, 10.2 / 8.7; 1 x 15,
// 4096: 17.2 / 14.3, 16.0 / 16.6.
static int column_parts_log2(int H, int D, int F, int B) {
  const int64_t groups = (int64_t)F * H;
  int parts = 0;
  if (D >= 128 && groups < 128) parts = 1;
  if (2 * D >> parts == 128 && groups <= 64 && groups % 8 == 0 && groups * B * D * 2 <= 17 << 20) ++parts;
  return parts;
}

// Whether a chunk's tokens go to one workgroup (a head's columns in parts or not), or to many in two stages.  Those for very
// many chunks of at most eight tokens per lane: whole rows of all heads, in the order they lie, then read faster than they add
// up (65536 tokens, 32 heads, chunk 128: 104 us in two stages, 114 in one; 8 heads: 28 and 22).  And where a workgroup would read
// so much that its chain outlasts them: beyond 2 MiB; for rows of all heads of less than 512 bytes, which the two stages handle
// faster, beyond 1 MiB, or 384 KiB unless there are many chunks.  Two stages / one, 128-element heads:
// 1 x 7, 3000: 15.0 / 13.6, 14.8 / 11.9; 1 x 3, 4096: 15.5 / 15.0, 18.3 / 14.5; 1 x 31, 4096: 20.9 / 20.4, 19.3 / 15.6; 1 x 3, 8192: 22.2 /
// 22.1, 28.9 / 22.5; 1 x 31, 8192: 32.0 / 31.8, 30.9 / 24.5; 2 x 3, 8192: 36.2 / 35.5, 30.9 / 22.6; 8 x 3, 8192: 44.7 / 48.2, 37.6 /
// 25.4; 1 x 3, 16384: 35.4 / 35.2, 51.6 / 38.2; 2 x 3, 16384: 64.9 / 64.3, 54.6 / 38.6; 4 x 1, 16384: 62.0 / 61.7, 67.6 / 40.9;
// 64-element heads: 1 x 7, 3000: 13.7 / 12.3, 14.2 / 11.6; 1 x 7, 4096: 13.4 / 13.0, 17.3 / 14.2; 1 x 63, 4096: 18.4 / 18.6, 18.2 / 15.3;
// 1 x 7, 8192: 16.4 / 16.2, 26.9 / 22.1; 4 x 7, 8192: 39.0 / 38.9, 31.8 / 23.0.
static bool whole_chunks(int H, int D, int F, int B) {
  const int d8 = D / 8;
  if (d8 > 16 || (d8 & (d8 - 1)) || H > 65535) return false;
  const int64_t groups = (int64_t)F * H;
  if (B * d8 <= 256 * 8 && groups > 8192) return false;
  if (groups >= 128) return true;
  const int parts_log2 = column_parts_log2(H, D, F, B);
  const int64_t bytes = (int64_t)B * D * 2 >> parts_log2;  // of a workgroup
  if (H * D >= 256) return bytes <= 2 << 20;
  return bytes <= 384 << 10 || (bytes <= 1 << 20 && (groups << parts_log2) * H * D > 30 * 128);
}

static int launch_chunk_mean(const void* k, const int32_t* fchunk_tok, void* kbar, double* partial, int H, int D,
                             int F, int B, int nsplit, int64_t kts, int64_t khs, int batch_rows, int64_t kbs, int dtype,
                             int* clear, int64_t clear_ints, hipStream_t st) {
  LaunchCheck launch_check;
  if (!partial) {  // (whole_chunks)
    int d8_log2 = 0;
    while ((8 << d8_log2) < D) ++d8_log2;
    const int parts_log2 = column_parts_log2(H, D, F, B);
    d8_log2 -= parts_log2;
    const dim3 grid(F, H, 1 << parts_log2);
    // threads: as many as eight tokens each would take, to be done soonest, or 256 where there are workgroups enough
    const int rows = (int64_t)F * H >= 1024 ? 256 : B * (D >> (3 + parts_log2)) / 8;
#define MOBA_MEAN(EL, NT)                                                                                                \
  hipLaunchKernelGGL((chunk_mean_whole_kernel<EL, NT>), grid, dim3(NT), 0, st, (const EL::elem*)k, fchunk_tok,            \
                     (EL::elem*)kbar, d8_log2, B, kts, khs, batch_rows, kbs, clear, clear_ints)
#define MOBA_MEAN_NT(EL)                          \
  if (rows <= 256) MOBA_MEAN(EL, 256);            \
  else if (rows <= 512) MOBA_MEAN(EL, 512);       \
  else MOBA_MEAN(EL, 1024)
    if (dtype == MOBA_DTYPE_F16) {
      MOBA_MEAN_NT(F16);
    } else {
      MOBA_MEAN_NT(Bf16);
    }
#undef MOBA_MEAN_NT
#undef MOBA_MEAN
    return launch_check.result();
  }
  const int HD8 = H * D / 8;
  const int tps = (B + nsplit - 1) / nsplit;
  const int cpb_log2 = pick_cpb_log2(HD8);
  dim3 grid(F, nsplit, (HD8 + (1 << cpb_log2) - 1) >> cpb_log2);
  const int64_t n = (int64_t)F * HD8;
  const dim3 fgrid((unsigned)((n + 63) / 64));
  if (dtype == MOBA_DTYPE_F16) {
    hipLaunchKernelGGL(chunk_mean_partial_kernel<F16>, grid, dim3(256), 0, st, (const f16*)k, fchunk_tok, partial,
                       HD8, D / 8, B, nsplit, tps, kts, khs, batch_rows, kbs, cpb_log2, clear, clear_ints);
    hipLaunchKernelGGL(chunk_mean_finish_kernel<F16>, fgrid, dim3(64), 0, st, (const double*)partial, (f16*)kbar,
                       HD8, B, nsplit, F);
  } else {
    hipLaunchKernelGGL(chunk_mean_partial_kernel<Bf16>, grid, dim3(256), 0, st, (const bf16*)k, fchunk_tok, partial,
                       HD8, D / 8, B, nsplit, tps, kts, khs, batch_rows, kbs, cpb_log2, clear, clear_ints);
    hipLaunchKernelGGL(chunk_mean_finish_kernel<Bf16>, fgrid, dim3(64), 0, st, (const double*)partial, (bf16*)kbar,
                       HD8, B, nsplit, F);
  }
  return launch_check.result();
}

// argument checks shared by the two entry points; kts, khs, kbr, kbs receive the key token and head strides, the
// rows per batch entry and the batch stride (elements)
static int check_chunk_mean_args(const void* k, const int32_t* fchunk_tok, void* kbar, int64_t S, int H, int D, int F,
                                 int B, const int64_t* strides, int dtype, int64_t& kts, int64_t& khs, int& kbr,
                                 int64_t& kbs) {
  if (dtype != MOBA_DTYPE_BF16 && dtype != MOBA_DTYPE_F16) return MOBA_ERR_UNSUPPORTED;
  if (!k || !fchunk_tok || !kbar || S <= 0 || H <= 0 || D <= 0 || F < 0 || B <= 0) return MOBA_ERR_ARG;
  if ((H * D) % 8 != 0 || ((uintptr_t)k & 15) || ((uintptr_t)kbar & 15)) return MOBA_ERR_ARG;
  if (D % 8 != 0) return MOBA_ERR_ARG;
  // strides (elements): {., ., k token, k head, rows per batch entry, ., k batch}; null = packed [S, H, D]
  kts = strides ? strides[2] : (int64_t)H * D;
  khs = strides ? strides[3] : D;
  if (strides && (strides[4] < 0 || strides[4] > 0x7fffffffLL)) return MOBA_ERR_ARG;  // (before it is narrowed)
  kbr = strides ? (int)strides[4] : 0;
  kbs = strides ? strides[6] : 0;
  if (kts <= 0 || khs <= 0 || (kts & 7) || (khs & 7)) return MOBA_ERR_ARG;
  if (kbr < 0 || (kbr > 0 && (kbs <= 0 || (kbs & 7)))) return MOBA_ERR_ARG;
  return MOBA_OK;
}

extern "C" int moba_chunk_mean(const void* k, const int32_t* fchunk_tok, void* kbar, void* workspace,
                               int64_t S, int H, int D, int F, int B, const int64_t* strides, int dtype,
                               int32_t* clear, int64_t clear_ints, void* stream) {
  if (clear_ints < 0 || (clear_ints > 0 && !clear)) return MOBA_ERR_ARG;
  if (F == 0) return MOBA_OK;  // (nothing to clear for: without chunks there are no lists to count)
  int64_t kts = 0, khs = 0, kbs = 0;
  int kbr = 0;
  const int rc = check_chunk_mean_args(k, fchunk_tok, kbar, S, H, D, F, B, strides, dtype, kts, khs, kbr, kbs);
  if (rc != MOBA_OK) return rc;
  if (!workspace || ((uintptr_t)workspace & 7)) return MOBA_ERR_ARG;
  double* partial = whole_chunks(H, D, F, B) ? nullptr : (double*)workspace;
  return launch_chunk_mean(k, fchunk_tok, kbar, partial, H, D, F, B, pick_nsplit(H * D / 8, F, B), kts, khs,
                           kbr, kbs, dtype, clear_ints > 0 ? clear : nullptr, clear_ints, (hipStream_t)stream);
}

// ---- the same stage for callers that cannot allocate: the partial sums live in a fixed array of the library ----
// Every GPU the library runs on holds its own copy of this array, at its own address, until the process
// ends.  The name below is a host-side stand-in, not a device address: host code only ever uses the
// address that hipGetSymbolAddress returned for the current device.
constexpr size_t kStaticPartialBytes = (size_t)32 << 20;
static __device__ __align__(256) double scratch[kStaticPartialBytes / sizeof(double)];

static std::mutex scratch_lock;
static double* scratch_of_device[kMaxDevices];   // guarded by scratch_lock

// device address of `scratch` on the current device (null on error), asked once per device
static double* static_partials() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return nullptr;
  std::lock_guard<std::mutex> hold(scratch_lock);
  if (dev < kMaxDevices && scratch_of_device[dev]) return scratch_of_device[dev];
  double* ptr = nullptr;
  if (hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return nullptr;
  if (dev < kMaxDevices) scratch_of_device[dev] = ptr;
  return ptr;
}

extern "C" size_t moba_chunk_mean_static_capacity(void) { return kStaticPartialBytes; }

extern "C" int moba_chunk_mean_static(const void* k, const int32_t* fchunk_tok, void* kbar, int64_t S, int H, int D,
                                      int F, int B, const int64_t* strides, int dtype, void* stream) {
  if (F == 0) return MOBA_OK;
  int64_t kts = 0, khs = 0, kbs = 0;
  int kbr = 0;
  const int rc = check_chunk_mean_args(k, fchunk_tok, kbar, S, H, D, F, B, strides, dtype, kts, khs, kbr, kbs);
  if (rc != MOBA_OK) return rc;
  // The sums are exact in fp64, so the mean does not depend on the number of token splits: take the
  // widest split (up to the one moba_chunk_mean would use) whose partial sums fit the array.
  const int HD8 = H * D / 8;
  const size_t per_split = (size_t)F * HD8 * 8 * sizeof(double);
  if (per_split > kStaticPartialBytes) return MOBA_ERR_LIMIT;   // F * H * D * 8 bytes exceed the array
  int nsplit = pick_nsplit(HD8, F, B);
  while (nsplit > 1 && per_split * nsplit > kStaticPartialBytes) nsplit /= 2;
  double* partial = nullptr;
  if (!whole_chunks(H, D, F, B)) {
    partial = static_partials();
    if (!partial) return MOBA_ERR_LAUNCH;
  }
  return launch_chunk_mean(k, fchunk_tok, kbar, partial, H, D, F, B, nsplit, kts, khs, kbr, kbs, dtype, nullptr, 0,
                           (hipStream_t)stream);
}
