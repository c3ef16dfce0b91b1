// Parameter-less gate and causal top-k.
//
// score(s, h, f) = <q[s,h,:], kbar[f,h,:]> in fp32 (bf16 x bf16 products are exact in
// fp32; the MFMA accumulates them in fp32).  A token s in the c-th chunk of its
// sequence may pick among the c earlier chunks of the same sequence, whose
// filtered-chunk ids are [fb, fb + c) with fb the first filtered id of the
// sequence.  The K best are kept; ties go to the lower chunk id; a -inf or NaN
// score is never picked.  Output sel[s, h, 0..K) holds filtered-chunk ids in
// descending score order, -1 padded.  With dense_local = d > 0 the tokens of the
// chunks 0..d of every sequence (which would pick every earlier chunk) get no picks
// at all: the attention kernels serve them through one causal pass over the prefix.
//
// One wave handles 64 consecutive tokens of one head (a workgroup four heads of them, or 256 tokens of one head: see
// by_tokens): the score tile (32 chunks x 64 tokens) is two 32x32x16 MFMA
// accumulators.  Sixteen lane-half swaps leave the 32 scores of token `lane` in lane `lane`; a lane marks those that
// beat the worst entry of its list (three instructions each, no LDS) and inserts them one per pass, lowest id first, in
// a top-k held in registers.  Scores never reach HBM (except through the optional debug output).
//
// Bound: Q is read once (HBM) for few candidates; with many the vector instructions per candidate decide.  Measured at
// 196608 tokens, 32 heads on 8, up to 767 candidates, 2 picks: 2.20 ms with the tile transposed through LDS and a
// barrier on either side of it, 1.39 ms here; 302060 tokens, up to 147 candidates: 1.12 -> 0.91 ms; 65536 tokens, 16
// heads, up to 511 candidates, 11 picks: 422 -> 333 us.  The first block stops at the last candidate (4096 tokens, 4 heads: 11.0 ->
// 10.1 us; 8191 tokens, 32 heads of 64: 23.8 -> 21.8).
#include <algorithm>
#include "common.h"

namespace moba {

template <int KMAX>
struct TopK {
  float val[KMAX];
  int idx[KMAX];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      val[j] = -INFINITY;
      idx[j] = -1;
    }
  }
  // keep the list sorted by descending value; an equal value stays behind the
  // entries already present, so among equal scores the lower id (seen first) wins
  // (the values are in descending order, so the new entry j is the median of the old entries j - 1 and j and of
  // x: one instruction; inside the test x is a number)
  __device__ __forceinline__ void push(float x, int id) {
    if (x > val[KMAX - 1]) {
#pragma unroll
      for (int j = KMAX - 1; j >= 1; --j) {
        const bool shift = x > val[j - 1];
        const bool here = x > val[j];
        idx[j] = shift ? idx[j - 1] : (here ? id : idx[j]);
        val[j] = __builtin_amdgcn_fmed3f(val[j - 1], val[j], x);
      }
      idx[0] = x > val[0] ? id : idx[0];
      val[0] = fmaxf(val[0], x);
    }
  }
};

// locate the sequence of token s: largest b with cu[b] <= s
__device__ __forceinline__ int find_seq(const int* __restrict__ cu, int nseq, int s) {
  return upper_row(cu, nseq, s);
}

// (up to 4 picks the kernel is held to the registers of three waves per SIMD, whose waves issue their vector
// instructions while others wait; longer lists would spill there: 11 picks, 31 candidates: 422 us held to three, 337 to
// two)
template <class E, int KMAX, int D>
__global__ __launch_bounds__(256, KMAX <= 4 || (KMAX <= 12 && D == 64) ? 3 : (KMAX <= 16 ? 2 : 1)) void gate_topk_kernel(
    const typename E::elem* __restrict__ q, const typename E::elem* __restrict__ kbar, const int* __restrict__ cu_seqlens,
    const int* __restrict__ seq_fbase, int* __restrict__ sel, float* __restrict__ scores_out,
    int S, int H, int Hkv, int nseq, int F, int B, int K, int64_t q_tok_stride, int64_t q_head_stride,
    int batch_rows, int64_t q_batch_stride, const int* __restrict__ pair_off, int* __restrict__ cnt, int dense_local,
    int one_head) {
  MOBA_ELEM_TYPES(E)
  // a lane's 32 scores, for the passes that take one of them by its number (rows 136 bytes apart: 8-byte writes, and reads of
  // one number by all lanes, spread over the banks); later the staged lists and the histograms
  __shared__ __attribute__((aligned(16))) float sc[4][64][34];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = lane & 31, hh = lane >> 5;
  const int tile = one_head ? blockIdx.x / H : blockIdx.x;  // (one_head: the heads of the same tokens side by side)
  const int tok0 = one_head ? tile * 256 + wave * 64 : tile * 64;
  const int h = one_head ? blockIdx.x - tile * H : blockIdx.y * 4 + wave;
  const bool head_ok = h < H;
  const int hc = head_ok ? h : H - 1;

  // this lane's own token (selection phase)
  const int s = tok0 + lane;
  int fb = 0, c = 0;
  if (s < S) {
    const int b = find_seq(cu_seqlens, nseq, s);
    fb = seq_fbase[b];
    c = (s - cu_seqlens[b]) / B;
    // a token of a dense prefix attends all its earlier chunks through the causal self path: no picks, no counts
    if (c <= dense_local) c = 0;
  }
  // union of the candidate ranges of the wave's 64 tokens (the same for the workgroup's other waves only where they hold other
  // heads of the same tokens: no barrier may stand under a test of them)
  int flo = c > 0 ? fb : 0x7fffffff;
  int fhi = c > 0 ? fb + c : 0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    flo = min(flo, __shfl_xor(flo, o, 64));
    fhi = max(fhi, __shfl_xor(fhi, o, 64));
  }

  TopK<KMAX> top;
  top.init();

  if (fhi > 0) {  // wave-uniform
    // Q^T operand: lane (n, hh) holds q[token n (+32)][16*ks + 8*hh .. +7]
    elem8 bq[2][D / 16];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const int tok = min(tok0 + 32 * qb + n, S - 1);
      const int be = batch_rows ? tok / batch_rows : 0;  // batch entry of the token in a batched layout
      const elem* src = q + (be * q_batch_stride + (tok - be * batch_rows) * q_tok_stride + hc * q_head_stride) + 8 * hh;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) bq[qb][ks] = *reinterpret_cast<const elem8*>(src + 16 * ks);
    }
    const elem* const kb_head = kbar + (hc / (H / Hkv)) * D + 8 * hh;
    elem8 a[D / 16];  // the chunk representatives of the block to come
    auto load_block = [&](int f0) __attribute__((always_inline)) {
      const elem* src = kb_head + (int64_t)min(f0 + n, F - 1) * Hkv * D;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) a[ks] = *reinterpret_cast<const elem8*>(src + 16 * ks);
    };
    constexpr bool kAhead = KMAX <= 16;  // (longer lists leave it no registers: 32 picks 400 us with it, 277 without)
    if constexpr (kAhead) load_block(flo);
    float* const mine = &sc[wave][lane][0];
    for (int f0 = flo; f0 < fhi; f0 += 32) {
      if constexpr (!kAhead) load_block(f0);
      f32x16 acc0 = {0}, acc1 = {0};
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        acc0 = mfma32(a[ks], bq[0][ks], acc0);
        acc1 = mfma32(a[ks], bq[1][ks], acc1);
      }
      if constexpr (kAhead) {
        if (f0 + 32 < fhi) load_block(f0 + 32);  // (travels while this block is gone through)
      }
      // Lane (n, hh) holds the scores of chunks 8*(e/4) + 4*hh + e%4 for tokens n (acc0) and 32 + n (acc1).  Swapping
      // acc1 of the lower half with acc0 of the upper one gives lane l token l: chunks 8*(e/4) + e%4 in acc0 and
      // 4 more than that in acc1.
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const auto r = __builtin_amdgcn_permlane32_swap(float_bits(acc0[e]), float_bits(acc1[e]), false, false);
        acc0[e] = __builtin_bit_cast(float, (uint32_t)r[0]);
        acc1[e] = __builtin_bit_cast(float, (uint32_t)r[1]);
      }
      auto score = [&](int j) __attribute__((always_inline)) {  // of chunk f0 + j (j a constant once unrolled)
        return (j & 4) ? acc1[4 * (j >> 3) + (j & 3)] : acc0[4 * (j >> 3) + (j & 3)];
      };
      const int lo = max(fb - f0, 0), hi = min(fb + c - f0, 32);  // chunks f0 + lo .. f0 + hi - 1 are the token's to pick
      auto to_lds = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          *reinterpret_cast<float2*>(mine + 8 * (g >> 1) + 2 * (g & 1)) = make_float2(acc0[2 * g], acc0[2 * g + 1]);
          *reinterpret_cast<float2*>(mine + 8 * (g >> 1) + 4 + 2 * (g & 1)) = make_float2(acc1[2 * g], acc1[2 * g + 1]);
        }
      };
      if (scores_out) {  // (uniform)
        to_lds();
        for (int j = lo; j < hi; ++j)
          if (head_ok) scores_out[((int64_t)s * H + h) * F + f0 + j] = mine[j];
      }
      if (f0 == flo) {  // (uniform) the first candidates: every one of them enters the list
        if constexpr (KMAX <= 16) {
#pragma unroll
          for (int j = 0; j < 32; ++j) {
            if ((j & 7) == 0 && f0 + j >= fhi) break;  // (wave-uniform)
            const float x = score(j);
            if (j >= lo && j < hi) top.push(x, f0 + j);
          }
        } else {  // (32 copies of a long insertion would not fit the instruction cache)
          to_lds();
#pragma unroll 4
          for (int j = 0; j < 32; ++j)
            if (j >= lo && j < hi) top.push(mine[j], f0 + j);
        }
        continue;
      }
      // the candidates that beat the list's worst entry as the block begins (it only rises), chunk f0 + j in bit 31 - j;
      // a -inf or NaN score beats nothing
      const float worst = top.val[KMAX - 1];
      uint32_t beat = 0;
#pragma unroll
      for (int j = 0; j < 32; ++j) beat = beat + beat + (score(j) > worst ? 1u : 0u);
      beat &= hi > lo ? (0xffffffffu >> lo) & (0xffffffffu << (32 - hi)) : 0u;
      if (!__ballot(beat != 0)) continue;  // (wave-uniform)
      to_lds();
      while (__ballot(beat != 0)) {  // (wave-uniform) one insertion per lane and pass, in ascending order of the ids
        if (beat) {
          const int j = __clz(beat);
          beat &= ~(0x80000000u >> j);
          top.push(mine[j], f0 + j);
        }
      }
    }
  }
  // The lists, K ints per (token, head): of four heads that lie side by side, 4K ints in a row per token in sel, or of one head,
  // K ints in a row every H * K.  Through LDS, so that the workgroup stores those runs with consecutive lanes on consecutive
  // ints (a lane storing its own K ints touches a cache line for 4K bytes of it).
  __syncthreads();  // (the score tile is read out)
  int* stage = reinterpret_cast<int*>(&sc[0][0][0]);  // [64 tokens][4 heads][K], or one_head: [256 tokens][K]
  if (4 * 64 * K <= (int)(sizeof(sc) / sizeof(int))) {  // (uniform; K <= 34)
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (j < K) stage[(one_head ? wave * 64 + lane : lane * 4 + wave) * K + j] = top.idx[j];
    __syncthreads();
    if (one_head) {
      const int first = tile * 256;
      for (int i = threadIdx.x; i < 256 * K; i += 256) {
        const int tk = i / K;
        if (first + tk < S) sel[((int64_t)(first + tk) * H + h) * K + i - tk * K] = stage[i];
      }
    } else {
      const int run = 4 * K;                       // ints per token in this workgroup's four heads
      const int heads_here = min(4, H - blockIdx.y * 4);
      for (int i = threadIdx.x; i < 64 * run; i += 256) {
        const int tk = i / run, w = i - tk * run;  // token of the tile, int within its run
        if (tok0 + tk < S && w < heads_here * K)
          sel[((int64_t)(tok0 + tk) * H + blockIdx.y * 4) * K + w] = stage[i];
      }
    }
  } else if (s < S && head_ok) {
    int* dst = sel + ((int64_t)s * H + h) * K;
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (j < K) dst[j] = top.idx[j];
  }
  // The gather lists' counts as a by-product: how many tokens of a (query chunk, head) picked each earlier chunk,
  // added into cnt[(chunk, head, query chunk)] (integer sums: the order of the additions does not matter).  A
  // wave's 64 tokens lie in one query chunk, or in a few: one pass per chunk, through a histogram in LDS of the wave's own, or
  // of all four waves' (one_head) where their tokens lie in one query chunk with up to 64 earlier ones.
  if (!cnt) return;
  constexpr int kHist = (int)(sizeof(sc) / sizeof(int)) / 4;
  int* const hists = reinterpret_cast<int*>(&sc[0][0][0]);
  const bool counts = head_ok && s < S && c > 0;
  uint64_t todo = __ballot(counts);
  int* hist = hists + wave * kHist;
  auto add_up = [&](int* hist, int cfb, int w0, int wn) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      const int i = (j < K && top.idx[j] >= 0) ? top.idx[j] - cfb - w0 : -1;
      if ((unsigned)i < (unsigned)wn) atomicAdd(&hist[i], 1);
    }
  };
  auto to_counts = [&](int n, int cc, int cfb, int at) __attribute__((always_inline)) {  // n picks of chunk cfb + at
    if (n == 0) return;  // (nearly all of many candidates: nothing is looked up for them)
    const int f = cfb + at;
    const int q0 = pair_off[f], nq = pair_off[f + 1] - q0;
    atomicAdd(&cnt[q0 * H + h * nq + (cc - at - 1)], n);
  };
  if (one_head) {
    // the four waves' tokens, if they lie in one query chunk: one histogram, one addition for each count where the waves on
    // their own make four (the additions of a call of few heads meet in a few cache lines)
    __shared__ int4 of_wave[4];
    const int leader = todo ? __ffsll((unsigned long long)todo) - 1 : 0;
    const int cc = __shfl(c, leader, 64), cfb = __shfl(fb, leader, 64);
    const bool same = __ballot(counts && c == cc && fb == cfb) == todo;
    if (lane == 0) of_wave[wave] = make_int4(todo != 0, cc, cfb, same);
    __syncthreads();  // (the staged lists are stored)
    const int4 w0 = of_wave[0];
    bool joint = w0.x != 0 && w0.y <= 64;
#pragma unroll
    for (int w = 0; w < 4; ++w) joint = joint && (of_wave[w].x != 0 && of_wave[w].y == w0.y && of_wave[w].z == w0.z && of_wave[w].w != 0);
    if (joint) {  // (block-uniform)
      if (threadIdx.x < 64) hists[threadIdx.x] = 0;
      __syncthreads();
      if (counts) add_up(hists, cfb, 0, cc);
      __syncthreads();
      if ((int)threadIdx.x < cc) to_counts(hists[threadIdx.x], cc, cfb, threadIdx.x);
      return;
    }
  } else {
    __syncthreads();  // (the staged lists are stored)
  }
  while (todo) {  // (wave-uniform)
    const int leader = __ffsll((unsigned long long)todo) - 1;
    const int cc = __shfl(c, leader, 64), cfb = __shfl(fb, leader, 64);
    const bool mine = counts && c == cc && fb == cfb;
    for (int w0 = 0; w0 < cc; w0 += kHist) {
      const int wn = min(kHist, cc - w0);
      for (int i = lane; i < wn; i += 64) hist[i] = 0;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (mine) add_up(hist, cfb, w0, wn);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int i = lane; i < wn; i += 64) to_counts(hist[i], cc, cfb, w0 + i);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    todo &= ~__ballot(mine);
  }
}

// Selection alone, on scores supplied by the caller ([S, H, F] fp32, -inf where a
// chunk is not a valid candidate).  Same insertion routine as the fused kernel.
template <int KMAX>
__global__ __launch_bounds__(256) void topk_from_scores_kernel(const float* __restrict__ scores,
                                                               int* __restrict__ sel, int64_t rows, int F, int K) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= rows) return;
  TopK<KMAX> top;
  top.init();
  const float* src = scores + r * F;
  for (int f = 0; f < F; ++f) top.push(src[f], f);
  int* dst = sel + r * K;
#pragma unroll
  for (int j = 0; j < KMAX; ++j)
    if (j < K) dst[j] = top.idx[j];
}

}  // namespace moba

using namespace moba;

#define MOBA_DISPATCH_K(K, CALL)            \
  if ((K) <= 2) { CALL(2); }                \
  else if ((K) <= 4) { CALL(4); }           \
  else if ((K) <= 8) { CALL(8); }           \
  else if ((K) <= 12) { CALL(12); }         \
  else if ((K) <= 16) { CALL(16); }         \
  else if ((K) <= 32) { CALL(32); }         \
  else if ((K) <= 64) { CALL(64); }         \
  else return MOBA_ERR_LIMIT;

// What a workgroup's four waves are: heads of the same 64 tokens, whose picks leave as one run per token, or 256 tokens of a head,
// whose counts leave as one addition.  By tokens in two cases; below by heads / by tokens in us, 2 picks, with the counts, one
// sequence, Q just written.
// Waves without a head, a twelfth of all and more, where the chip's 1024 SIMDs have no room for them beside the others at a wave
// each.  Chunk 128: one head, 16379 tokens: 15.6 / 15.4; 24571: 22.1 / 18.3; 262139: 541 / 179; 2 heads, 16379: 15.8 / 16.0; 24571: 22.2 /
// 19.1; 3 heads, 16379: 16.4 / 16.8; 21840: 22.2 / 19.4; 5 heads, 52423: 80.4 / 56.1; 13 heads, 20159: 45.6 / 37.7; 22 heads, 2508: 11.5 /
// 12.2; 2880: 13.5 / 12.4; 11910: 35.8 / 32.7.
// The additions.  A counter gets one from each wave of its query chunk, B / 64 by heads and a quarter of that by tokens, and a
// kernel of up to a wave to a SIMD waits for them at its end; with 4 heads, whose counters lie in few cache lines, longer ones
// with long chunks do too.  Chunks of less than 512 tokens have nothing to gain: a workgroup's tokens then lie in two of them
// as often as not.  8 heads, 8187 tokens, chunk 128: 13.8 / 14.9; 256: 12.4 / 12.8; 512: 12.3 / 11.9; 2048: 15.9 / 11.6; 4 heads, 32763
// tokens, 512: 18.6 / 17.8; 2048: 22.4 / 15.5; 65531, 512: 32.6 / 34.0; 2048: 30.9 / 24.6.  More rows of more heads gain with long chunks
// of one sequence (8 heads, 16379 tokens, 2048: 20.7 / 14.6) and may lose with several (16 heads, 3 x 5457, 4096, Q from memory: 15.9 /
// 18.3): by heads.
static bool by_tokens(int64_t S, int H, int B) {
  const int64_t heads = (H + 3) / 4 * 4ll;  // with those that waves have none for
  if ((heads - H) * 12 >= heads && (S + 63) / 64 * heads > 1024) return true;
  return B >= 512 && S * H <= (H == 4 ? std::max<int64_t>(65536, 256ll * B) : 65536);
}

extern "C" int moba_gate_topk(const void* q, const void* kbar, const int32_t* cu_seqlens, const int32_t* seq_fbase,
                              int32_t* sel, float* scores_out, const int32_t* pair_off, int32_t* cnt, int64_t S, int H,
                              int Hkv, int D, int nseq, int F, int B, int K, int dense_local, const int64_t* strides,
                              int dtype, void* stream) {
  LaunchCheck launch_check;
  if (!q || !kbar || !cu_seqlens || !seq_fbase || !sel || (cnt && !pair_off)) return MOBA_ERR_ARG;
  if (Hkv <= 0 || H % Hkv != 0) return MOBA_ERR_ARG;
  if (dtype != MOBA_DTYPE_BF16 && dtype != MOBA_DTYPE_F16) return MOBA_ERR_UNSUPPORTED;
  if (S <= 0 || S > 0x7fffffff - 64 || H <= 0 || nseq <= 0 || F <= 0 || B <= 0 || K <= 0) return MOBA_ERR_ARG;
  if (dense_local < 0 || dense_local > K) return MOBA_ERR_ARG;
  if (D != kHeadDim && D != 64) return MOBA_ERR_UNSUPPORTED;
  if (((uintptr_t)q & 15) || ((uintptr_t)kbar & 15)) return MOBA_ERR_ARG;
  // strides (elements): {q token, q head, ., ., rows per batch entry, q batch, .}; null = packed [S, H, D]
  const int64_t qts = strides ? strides[0] : (int64_t)H * D, qhs = strides ? strides[1] : D;
  if (strides && (strides[4] < 0 || strides[4] > 0x7fffffffLL)) return MOBA_ERR_ARG;  // (before it is narrowed)
  const int qbr = strides ? (int)strides[4] : 0;
  const int64_t qbs = strides ? strides[5] : 0;
  if (qts <= 0 || qhs <= 0 || (qts & 7) || (qhs & 7)) return MOBA_ERR_ARG;
  if (qbr < 0 || (qbr > 0 && (qbs <= 0 || (qbs & 7)))) return MOBA_ERR_ARG;
  const int one_head = by_tokens(S, H, B);
  dim3 grid((unsigned)((S + 63) / 64), (unsigned)((H + 3) / 4));
  if (one_head) grid = dim3((unsigned)((S + 255) / 256 * H));
  hipStream_t st = (hipStream_t)stream;
#define GATE(EL, KM, DIM)                                                                                             \
  hipLaunchKernelGGL((gate_topk_kernel<EL, KM, DIM>), grid, dim3(256), 0, st, (const EL::elem*)q, (const EL::elem*)kbar, \
                     cu_seqlens, seq_fbase, sel, scores_out, (int)S, H, Hkv, nseq, F, B, K, qts, qhs, qbr, qbs,       \
                     pair_off, cnt, dense_local, one_head)
#define CALL(KM)                                                       \
  if (dtype == MOBA_DTYPE_F16) {                                       \
    if (D == 64) GATE(F16, KM, 64); else GATE(F16, KM, 128);           \
  } else {                                                             \
    if (D == 64) GATE(Bf16, KM, 64); else GATE(Bf16, KM, 128);         \
  }
  MOBA_DISPATCH_K(K, CALL)
#undef CALL
#undef GATE
  return launch_check.result();
}

extern "C" int moba_topk_from_scores(const float* scores, int32_t* sel, int64_t S, int H, int F, int K,
                                     void* stream) {
  LaunchCheck launch_check;
  if (!scores || !sel || S <= 0 || H <= 0 || F <= 0 || K <= 0) return MOBA_ERR_ARG;
  const int64_t rows = S * H;
  dim3 grid((unsigned)((rows + 255) / 256));
  hipStream_t st = (hipStream_t)stream;
#define CALL(KM) \
  hipLaunchKernelGGL(topk_from_scores_kernel<KM>, grid, dim3(256), 0, st, scores, sel, rows, F, K)
  MOBA_DISPATCH_K(K, CALL)
#undef CALL
  return launch_check.result();
}
