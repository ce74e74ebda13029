// Token sampler for gfx950: the step after the last layer's decode.
//
// A row's work, over passes of 1,024-thread workgroups (8 logits per thread and
// chunk; the row is L2 / MALL resident after the first pass):
//   x_i = (repetition penalty on seen tokens)(logit_i) / T   (T = 1 for greedy rows)
//   min_p:  keep x_i >= max + ln(min_p)             (p_i >= min_p * p_max)
//   top_k:  keep the k largest (ties kept), exact over order-preserving 32-bit keys
//   top_p:  keep token i iff the mass strictly above it is < top_p * mass
//           (64-bit fixed-point masses: integer sums, so the threshold is deterministic)
//   sample: argmax over kept i of x_i - ln(E_i), E_i ~ Exp(1) from a
//           counter-based hash of (seed, step, i) -- the exponential race,
//           an exact draw from softmax over the kept set; greedy rows take
//           argmax x_i. Ties go to the lowest index.
// Outputs: the token, its processed logprob (log-softmax over the kept set of
// the processed logits), the kept set as a bitmap and its size.
//
// One workgroup per row (sample_kernel) fills the chip from about 128 rows on.
// Fewer rows that are drawn from the whole vocabulary (no top_k, top_p or
// min_p), with a workspace, are cut into slices: sample_max_kernel (the
// slices' maxima), sample_slice_kernel (each slice's part of the draw) and
// sample_join_kernel, which joins the slices of a row.
#include <cmath>
#include <type_traits>

#include "wkv_common.h"

namespace wkv {

constexpr int kSampleThreads = 1024;
constexpr float kGreedyEps = 1e-5f;  // temperatures below this sample greedily
// A score x - ln E is at most x + 16.636 (u <= 1 - 2^-24): a token more than
// kScoreReach below a score already drawn never wins the race (0.064 of margin
// for float rounding).
constexpr float kScoreReach = 16.7f;

// Order-preserving key of a float (larger float -> larger key); NaN maps below
// every real value so it is never kept.
__device__ __forceinline__ uint32_t order_key(float x) {
  if (x != x) return 0u;
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// splitmix64 finaliser.
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// ln(E) of the Exp(1) variate of token i: u in [2^-24, 1 - 2^-24] from 23
// hash bits, exact in float32 (24 bits would round the top value to 1.0:
// E = 0 and an infinite race score for one token in 2^24). Both logarithms
// take the hardware log2 times ln 2: their arguments (u >= 2^-24, -ln u >=
// 6e-8) are never denormal, so logf's scaling and extended-precision fixups
// buy at most an ulp here.
__device__ __forceinline__ float log_exp_variate(uint64_t stream, int64_t i) {
  const uint64_t h = mix64(stream + static_cast<uint64_t>(i));
  // u = (m + 0.5) 2^-23 for the top 23 bits m, exactly: 1 + m 2^-23 from the
  // bits, minus 1 (exact), plus 2^-24 (exact at that magnitude).
  const uint32_t m = static_cast<uint32_t>(h >> 32) >> 9;
  const float u = (__uint_as_float(0x3F800000u | m) - 1.0f) + 5.9604644775390625e-8f;
  constexpr float kLn2 = 0.693147180559945309f;
  return __builtin_amdgcn_logf(-__builtin_amdgcn_logf(u) * kLn2) * kLn2;
}

template <typename T>
__device__ __forceinline__ float load_logit(const T *row, int64_t i);
template <>
__device__ __forceinline__ float load_logit<float>(const float *row, int64_t i) { return row[i]; }
template <>
__device__ __forceinline__ float load_logit<uint16_t>(const uint16_t *row, int64_t i) {
  return bf16_bits_to_f32(row[i]);
}

// Elements per thread per step: 8 consecutive logits, one or two 16-byte loads
// (of any element alignment: a row may start anywhere); -inf past the end.
constexpr int kVec = 8;
// Tokens one step of a workgroup covers.
constexpr int kStep8 = kSampleThreads * kVec;
// Chunks whose loads a pass issues together, one batch ahead of its use (with
// one 16-byte load per thread at a time a pass over a row is bound by the load
// latency, not by HBM). 64 bytes per thread and batch, two batches live.
template <typename T>
constexpr int batch_chunks() {
  return sizeof(T) == 2 ? 4 : 2;
}

// One chunk's raw bits: 16 bytes of bf16, or 32 of fp32.
template <typename T>
struct Chunk;
template <>
struct Chunk<uint16_t> {
  u32x4 w;
};
template <>
struct Chunk<float> {
  floatx4 a, b;
};

template <typename T>
__device__ __forceinline__ Chunk<T> load_chunk(const T *p) {
  if constexpr (sizeof(T) == 2) {
    typedef u32x4 __attribute__((aligned(2))) u32x4_a2;
    return Chunk<T>{*reinterpret_cast<const u32x4_a2 *>(p)};
  } else {
    typedef floatx4 __attribute__((aligned(4))) floatx4_a4;
    return Chunk<T>{*reinterpret_cast<const floatx4_a4 *>(p), *reinterpret_cast<const floatx4_a4 *>(p + 4)};
  }
}

template <typename T>
__device__ __forceinline__ void unpack_chunk(const Chunk<T> &c, float v[kVec]) {
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[2 * j] = __uint_as_float(c.w[j] << 16);
      v[2 * j + 1] = __uint_as_float(c.w[j] & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = c.a[j];
      v[4 + j] = c.b[j];
    }
  }
}

template <typename T>
__device__ __forceinline__ void load8(float v[kVec], const T *row, int64_t base, int vocab) {
  if (base + kVec <= vocab) {
    unpack_chunk<T>(load_chunk<T>(row + base), v);
  } else {
#pragma unroll
    for (int j = 0; j < kVec; ++j) v[j] = base + j < vocab ? load_logit<T>(row, base + j) : -INFINITY;
  }
}

// Block-wide reductions over 1024 threads (16 waves) through a small LDS array.
__device__ __forceinline__ float block_max(float v, float *red) {
  v = wave_max(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float r = red[0];
  for (int i = 1; i < kSampleThreads / 64; ++i) r = fmaxf(r, red[i]);
  __syncthreads();
  return r;
}

__device__ __forceinline__ float block_sum(float v, float *red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < kSampleThreads / 64; ++i) r += red[i];  // fixed order: deterministic
  __syncthreads();
  return r;
}

// (value, index) argmax, ties to the lowest index.
__device__ __forceinline__ void arg_better(float &v, int64_t &i, float ov, int64_t oi) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}

__device__ __forceinline__ void wave_argmax(float &v, int64_t &idx) {
  const auto step = [&](auto o) {
    constexpr int O = decltype(o)::value;
    arg_better(v, idx, lane_xor<O>(v), lane_xor<O>(idx));
  };
  step(std::integral_constant<int, 32>{});
  step(std::integral_constant<int, 16>{});
  step(std::integral_constant<int, 8>{});
  step(std::integral_constant<int, 4>{});
  step(std::integral_constant<int, 2>{});
  step(std::integral_constant<int, 1>{});
}

__device__ __forceinline__ void block_argmax(float &v, int64_t &idx, float *redv, int64_t *redi) {
  wave_argmax(v, idx);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    redv[w] = v;
    redi[w] = idx;
  }
  __syncthreads();
  v = redv[0];
  idx = redi[0];
  for (int i = 1; i < kSampleThreads / 64; ++i) arg_better(v, idx, redv[i], redi[i]);
  __syncthreads();
}

// 64-bit sums and scans over a wave and the 1024-thread block.
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
  return wave_reduce(v, [](unsigned long long a, unsigned long long b) { return a + b; });
}

__device__ __forceinline__ unsigned long long wave_incl_scan_u64(unsigned long long v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(v, o, 64);
    if (lane >= o) v += y;
  }
  return v;
}

// Exclusive scan of one value per thread in thread order; `total` gets the sum.
__device__ __forceinline__ unsigned long long block_exscan_u64(unsigned long long v, unsigned long long *red,
                                                               unsigned long long &total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long incl = wave_incl_scan_u64(v, lane);
  if (lane == 63) red[w] = incl;
  __syncthreads();
  unsigned long long before = 0, all = 0;
  for (int i = 0; i < kSampleThreads / 64; ++i) {
    if (i < w) before += red[i];
    all += red[i];
  }
  __syncthreads();
  total = all;
  return before + incl - v;
}

// Radix-select step on a 256-bin histogram, searched from the top bin down:
// the largest j with above + sum(hist[j..255]) >= target, and the sum
// strictly above it (bin -1 when no j qualifies). Wave 0 computes it (four
// bins per lane and one wave scan) and writes it to *bin_out / *cum_out.
__device__ __forceinline__ void find_from_top(const unsigned long long *hist, unsigned long long above,
                                              unsigned long long target, uint32_t *bin_out,
                                              unsigned long long *cum_out) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  unsigned long long h[4], s = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    h[q] = hist[255 - 4 * lane - q];
    s += h[q];
  }
  unsigned long long c = above + wave_incl_scan_u64(s, lane) - s;  // mass of the bins above this lane's
  int bin = -1;
  unsigned long long cum = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (bin < 0 && c + h[q] >= target) {
      bin = 255 - 4 * lane - q;
      cum = c;
    }
    c += h[q];
  }
  const unsigned long long hit = __ballot(bin >= 0);
  if (hit == 0ull) {
    if (lane == 0) *bin_out = 0xffffffffu;
  } else if (lane == __ffsll(static_cast<long long>(hit)) - 1) {
    *bin_out = static_cast<uint32_t>(bin);
    *cum_out = cum;
  }
}

// Fast top_k / top_p. Every kept token the threshold can keep lies within a
// range below the row maximum known after the first pass (top_k: the bin of
// the k-th largest of the threads' maxima; top_p alone: a bound on the tail's
// weight), and at most kCand kept tokens in that range go to an LDS list: the
// exact selects run over the list, and the draw, mass and mask come from it.
// With top_k (k <= 1,024) or min_p alone the range is narrow, and the first
// pass's maxima of every thread's groups of four chunks say where its tokens
// are: only those groups are read again (top_k 50 over 151,936 bf16 logits,
// 256 rows: 47 -> 30 us against a second pass over the row). top_p alone needs
// the whole row's mass, so its capture is a pass. Rows whose range holds more
// tokens take a histogram of the kept tokens by distance below the maximum
// (kBins bins of 1/kBinScale, the last one open-ended), whose block scan gives
// the threshold's bin, and a compaction pass of the kept tokens at or above
// it. Binning is monotone in the value, so the list holds every token the
// threshold can keep and the selects give the same keys as over the whole row;
// rows whose threshold still falls in the open bin or overflows the list take
// the full-row radix passes.
constexpr int kBins = 2048;
constexpr float kBinScale = 32.f;
constexpr int kCand = 4096;
// A token this many bins or more below the maximum (22.2 nats) weighs under
// one unit of fixed_mass: exactly 0.
constexpr int kMassBins = 711;
// Mask words that the list path builds in LDS at a time (longer rows take turns).
constexpr int kMaskWords = 8192;
// A thread's groups: 2^kGroupShift chunks each up to 262,144 tokens, doubled
// for longer rows until kGroups of them cover the row (300,000 bf16 tokens, 1 /
// 256 rows, against whole passes: top_k 50 with top_p 81.9 / 101.4 -> 26.7 /
// 39.6 us, min_p 46.0 / 61.7 -> 21.0 / 34.5).
constexpr int kGroups = 8, kGroupShift = 2;
// More chunks to read again than this under min_p (of up to kGroups x 1,024
// groups): a pass over the row is as cheap.
constexpr int kMaxHitChunks = 8192;
// Entries of a list whose thresholds are found by ranking: top_k and top_p
// together, or one of them, for which the radix select runs once (8,000 tokens,
// 128 rows, top_k 200: 22.0 us ranked, 18.8 by radix; top_k 20: 16.6 and 18.0).
constexpr int kRanked = 256, kRankedOne = 128;
// Draws a wave may hold back before making them 64 at a time: the final pass's
// fast loop makes them after every fourth token slot, so fewer than 64 pending
// and 64 per slot (its general loop holds fewer than 128).
constexpr int kFastQueue = 64 + 4 * 64;
static_assert(kBins == 2 * kSampleThreads, "the threshold scan gives every thread two bins");

// e^(x - mx) in units of 2^-32, truncated; x <= mx, so at most 2^32. (An
// infinite maximum, where x - mx is NaN, weighs what a finite one does; every
// other token of its row then weighs 0.)
__device__ __forceinline__ unsigned long long fixed_mass(float x, float mx) {
  const float v = expf(x - mx) * 4294967296.f;
  return v < 4294967296.f ? static_cast<unsigned long long>(static_cast<uint32_t>(v)) : 1ull << 32;
}

struct SampleArgs {
  const float *temperature;  // [B] or NULL (1.0)
  const int32_t *top_k;      // [B] or NULL; <= 0 or >= vocab: off
  const float *top_p;        // [B] or NULL; >= 1: off
  const float *min_p;        // [B] or NULL; <= 0: off
  const float *rep_penalty;  // [B] or NULL; 1: off
  const uint32_t *seen;      // [B, words] bitmap of prompt/output tokens or NULL
  const uint64_t *seeds;     // [B] or NULL (0)
  int64_t step;              // mixed into every row's random stream
  int64_t *tokens;           // [B]
  float *logprobs;           // [B] or NULL
  uint32_t *mask;            // [B, words] or NULL
  int32_t *counts;           // [B] or NULL
  int group_shift;           // log2 of the chunks of a thread's group (sample_kernel)
};

// Rows cut into S slices of `slice` tokens (a multiple of kStep8): what the
// slices of one row leave for each other, in the caller's workspace.
constexpr int kMaxSlices = 32;
constexpr int kSliceRows = 128;     // at most this many rows are cut,
constexpr int kMinSliceGain = 5;    // where a slice is at least this many chunks shorter than the row
struct SliceRow {
  float vmax[kMaxSlices];     // a slice's maximum
  float score[kMaxSlices];    // the best race score of its threads' maxima
  float z[kMaxSlices];        // its kept mass,
  float best[kMaxSlices];     // its winner's score,
  int32_t win[kMaxSlices];    // the winner,
  int32_t cnt[kMaxSlices];    // and kept tokens
};
struct Slices {
  SliceRow *rows;
  int S, slice;
};

// A row's processed logits.
template <typename T>
struct Row {
  const T *row;
  int vocab;
  const uint32_t *seen;  // NULL: no penalty
  float pen, inv_t;
  bool greedy;

  __device__ __forceinline__ Row(const T *logits, int64_t row_stride, int v, const SampleArgs &a, int b) {
    row = logits + static_cast<int64_t>(b) * row_stride;
    vocab = v;
    const float temp = a.temperature ? a.temperature[b] : 1.f;
    greedy = temp < kGreedyEps;
    inv_t = greedy ? 1.f : 1.f / temp;
    pen = a.rep_penalty ? a.rep_penalty[b] : 1.f;
    seen = (a.seen && pen != 1.f) ? a.seen + static_cast<int64_t>(b) * ((v + 31) / 32) : nullptr;
  }
  __device__ __forceinline__ float x_of(int64_t i) const {
    float l = load_logit<T>(row, i);
    if (seen && ((seen[i >> 5] >> (i & 31)) & 1u)) l = l > 0.f ? l / pen : l * pen;
    return l * inv_t;
  }
  // The 8 processed logits at base .. base+7 (base a multiple of 8 below vocab; -inf past the end).
  __device__ __forceinline__ void processed(float v[kVec], int64_t base) const {
    if (seen) {
      const uint32_t w = seen[base >> 5] >> (base & 31);  // one word
#pragma unroll
      for (int j = 0; j < kVec; ++j)
        if ((w >> j) & 1u) v[j] = v[j] > 0.f ? v[j] / pen : v[j] * pen;
    }
    if (inv_t != 1.f) {  // uniform (the RL default is temperature 1: two instructions less per token and pass)
#pragma unroll
      for (int j = 0; j < kVec; ++j) v[j] *= inv_t;
    }
  }
  __device__ __forceinline__ void x8(float v[kVec], int64_t base) const {
    load8<T>(v, row, base, vocab);
    processed(v, base);
  }
  // f(v, base) over this thread's chunks of tokens [lo, hi) in row order (lo a
  // multiple of kStep8, hi one or the vocabulary), NB chunks per batch and the
  // next batch's loads in flight. With EVERY f also sees the chunks past the
  // end (all -inf), so every lane of a wave makes the same calls. The loop
  // body is unrolled NB times: heavy passes take NB = 2 (the final pass's
  // draw code in eight copies ran 6% slower).
  template <int NB, class EVERY, class F>
  __device__ __forceinline__ void for_chunks(EVERY, int64_t lo, int64_t hi, F &&f) const {
    constexpr int64_t step = static_cast<int64_t>(NB) * kStep8;
    const int64_t t = static_cast<int64_t>(threadIdx.x) * kVec;
    Chunk<T> r[NB], nx[NB];
    auto fetch = [&](Chunk<T>(&q)[NB], int64_t c0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int64_t base = c0 + t + u * kStep8;
        if (base + kVec <= hi) q[u] = load_chunk<T>(row + base);
      }
    };
    fetch(r, lo);
    for (int64_t c0 = lo; c0 < hi; c0 += step) {
      if (c0 + step < hi) fetch(nx, c0 + step);  // uniform
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (c0 + u * kStep8 >= hi) break;  // uniform
        const int64_t base = c0 + t + u * kStep8;
        if (!EVERY::value && base >= hi) continue;
        float v[kVec];
        if (base + kVec <= hi) {
          unpack_chunk<T>(r[u], v);
          processed(v, base);
        } else if (base < hi) {
          x8(v, base);
        } else {
#pragma unroll
          for (int j = 0; j < kVec; ++j) v[j] = -INFINITY;
        }
        f(v, base);
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) r[u] = nx[u];
    }
  }
};
using Every = std::true_type;
using Own = std::false_type;

__device__ __forceinline__ float max8(const float v[kVec]) {  // NaN never wins
  return fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7])));
}

// This thread's maximum over tokens [lo, hi) and where it is: the pass keeps
// the chunk (a compare per chunk, not per token), whose tokens are read again.
template <typename T>
__device__ __forceinline__ int track_max(const Row<T> &row, int64_t lo, int64_t hi, float &tmx) {
  int64_t at = -1;
  row.template for_chunks<batch_chunks<T>()>(Own{}, lo, hi, [&](const float v[kVec], int64_t base) __attribute__((always_inline)) {
    const float m = max8(v);
    if (m > tmx) {
      tmx = m;
      at = base;
    }
  });
  if (at < 0) return 0;
  float v[kVec];
  row.x8(v, at);
  int j = kVec - 1;
#pragma unroll
  for (int i = kVec - 2; i >= 0; --i) j = v[i] == tmx ? i : j;
  return static_cast<int>(at) + j;
}

// min_p (and finiteness) as a key threshold: x >= max + ln(min_p); the maximum itself is always kept.
__device__ __forceinline__ uint32_t min_key(float mp, float mx) {
  uint32_t key_lo = order_key(-3.402823466e38f);  // finite values only
  if (mp > 0.f) {
    uint32_t k = order_key(mx + logf(mp));
    if (k > order_key(mx)) k = order_key(mx);  // min_p above 1 still keeps the maximum
    key_lo = k > key_lo ? k : key_lo;
  }
  return key_lo;
}

// The fixed-point mass top_p must reach (at least one unit: the maximum stays whatever top_p is).
__device__ __forceinline__ unsigned long long top_p_target(float tp, unsigned long long total) {
  const unsigned long long t =
      static_cast<unsigned long long>(ceil(static_cast<double>(tp) * static_cast<double>(total)));
  return t > 0ull ? t : 1ull;
}

// Bins below the maximum that hold every token top_p alone can keep: tokens
// more than r = ln(vocab / (1 - top_p)) + 1 below the maximum weigh at most
// (1 - top_p) / e of the maximum's weight all together, so the mass above the
// threshold is reached within r (the maximum's fixed-point weight is exactly
// 2^32, whence the kept mass is at least that).
__device__ __forceinline__ int top_p_bins(float tp, int vocab) {
  const double tail = 1.0 - static_cast<double>(tp);
  if (tail <= 1e-6) return kBins - 1;
  const double r = (log(static_cast<double>(vocab) / tail) + 1.0) * static_cast<double>(kBinScale);
  return r < static_cast<double>(kBins - 1) ? static_cast<int>(ceil(r)) : kBins - 1;
}

__device__ __forceinline__ uint64_t row_stream(const SampleArgs &a, int b) {
  return mix64((a.seeds ? a.seeds[b] : 0ull) + static_cast<uint64_t>(a.step) * 0x9E3779B97F4A7C15ull);
}

// The race of one thread: best score so far, and the bound below which a
// token cannot win (raised by the thread's own draws as they come: a token
// below bound - kScoreReach cannot reach it, so its draw is skipped).
constexpr int64_t kNoToken = 0x7fffffffffffffffll;
struct Race {
  bool greedy;
  uint64_t stream;
  float lim;
  float best = -INFINITY;
  int64_t bi = kNoToken;
  __device__ __forceinline__ void draw(float x, int64_t t) {  // not of greedy rows
    if (x >= lim) {
      arg_better(best, bi, x - log_exp_variate(stream, t), t);
      lim = fmaxf(lim, best - kScoreReach);
    }
  }
  __device__ __forceinline__ void run(float x, int64_t t) {
    if (greedy)
      arg_better(best, bi, x, t);
    else
      draw(x, t);
  }
};

// Final pass over tokens [lo, hi): the kept mass (this thread's share of e^(x -
// max)), the mask words, the kept count and the race (not of greedy rows whose
// winner pass 1 found: race.bi is then set). qx / qt: the wave's draw queue
// (kFastQueue values and tokens). Every lane makes the same calls (chunks past
// the end are all -inf, kept nowhere): the mask words are assembled across lanes.
template <typename T>
__device__ __forceinline__ void final_pass(const Row<T> &row, int64_t lo, int64_t hi, uint32_t key_lo, float mx,
                                           Race &race, float *qx, int32_t *qt, uint32_t *mask_row, float &z,
                                           int &cnt) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int words = (row.vocab + 31) / 32;
  int qn = 0;  // wave-uniform
  auto put = [&](bool c, unsigned long long bal, float x, int64_t t) __attribute__((always_inline)) {
    if (c) {
      const int at = qn + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                              static_cast<uint32_t>(bal >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bal), 0u)));
      qx[at] = x;
      qt[at] = static_cast<int32_t>(t);
    }
    qn += __popcll(bal);
  };
  auto draw = [&](int at) __attribute__((always_inline)) { race.draw(qx[at], qt[at]); };
  auto write_mask = [&](uint32_t bits, int64_t base) __attribute__((always_inline)) {
    cnt += __popc(bits);
    if (mask_row != nullptr) {
      // four consecutive lanes hold the 32 bits of one mask word
      const uint32_t b1 = __shfl_down(bits, 1, 64), b2 = __shfl_down(bits, 2, 64), b3 = __shfl_down(bits, 3, 64);
      const int64_t wd = base >> 5;
      if ((tid & 3) == 0 && wd < words) mask_row[wd] = bits | (b1 << 8) | (b2 << 16) | (b3 << 24);
    }
  };
  const bool won = row.greedy && race.bi != kNoToken;
  if ((!row.greedy || won) && key_lo < 0x80000000u) {
    // Fast loop: the keep threshold is a negative float t (the RL defaults
    // keep every finite token, and most min_p rows land here). Keys order
    // negative floats (-0 included) as the floats do and every non-negative
    // float above them, and NaN fails both compares as it fails the key test,
    // so: kept <=> v >= t, and a race candidate (kept and v >= lim) <=> v >=
    // max(t, lim), one float compare each. A chunk none of whose lanes keeps a
    // token, or has a candidate, is passed over by its maximum. The draws go
    // through a queue per wave, made 64 at a time after every fourth token
    // slot (lim only moves there): the token slots in between carry no draw
    // code, and the mass, counts and mask come out as in the general loop.
    const float thr = __uint_as_float(~key_lo);
    float clim = fmaxf(thr, race.lim);
    auto pass = [&](auto drawn) __attribute__((always_inline)) {  // (one instance with the race, one without)
    constexpr bool DRAWN = decltype(drawn)::value;
    row.template for_chunks<2>(Every{}, lo, hi, [&](const float v[kVec], int64_t base) __attribute__((always_inline)) {
      uint32_t bits = 0;
      const float m = max8(v);
      if (__ballot(m >= thr) != 0ull) {  // uniform
        const bool draws = DRAWN && __ballot(m >= clim) != 0ull;  // uniform
        // Every token of the wave's chunk is kept (the usual chunk of the RL
        // defaults): the least of them is at least thr, and no NaN reached the sum.
        float mn = fminf(fminf(fminf(v[0], v[1]), fminf(v[2], v[3])), fminf(fminf(v[4], v[5]), fminf(v[6], v[7])));
        float e = 0.f;
#pragma unroll
        for (int j = 0; j < kVec; ++j) e += __expf(v[j] - mx);
        if (__ballot(!(mn >= thr && e == e)) == 0ull) {  // uniform
          bits = 0xffu;
          z += e;
        } else {
#pragma unroll
          for (int j = 0; j < kVec; ++j) {
            const bool kept = v[j] >= thr;
            bits |= kept ? 1u << j : 0u;
            z += kept ? __expf(v[j] - mx) : 0.f;
          }
        }
        if (draws) {
#pragma unroll
          for (int j = 0; j < kVec; ++j) {
            const bool c = v[j] >= clim;
            const unsigned long long bal = __ballot(c);
            if (bal != 0ull) put(c, bal, v[j], base + j);  // uniform
            if ((j & 3) == 3) {
              while (qn >= 64) {  // uniform
                qn -= 64;
                draw(qn + lane);
              }
              clim = fmaxf(thr, race.lim);
            }
          }
        }
      }
      write_mask(bits, base);
    });
    };
    if (won)
      pass(std::false_type{});
    else
      pass(std::true_type{});
  } else {
    // The draws go through the queue too, one per lane: a draw taken in place
    // would hold the whole wave whenever any one lane needs it.
    row.template for_chunks<2>(Every{}, lo, hi, [&](const float v[kVec], int64_t base) __attribute__((always_inline)) {
      uint32_t bits = 0;
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        const bool kept = order_key(v[j]) >= key_lo;
        if (__ballot(kept) == 0ull) continue;  // uniform: nothing kept in this slot of the wave
        if (kept) {
          bits |= 1u << j;
          z += __expf(v[j] - mx);  // (relative error ~1e-6 at 100 below the maximum)
        }
        if (row.greedy) {
          if (kept) arg_better(race.best, race.bi, v[j], base + j);  // (a winner of pass 1 stays)
          continue;
        }
        const bool c = kept && v[j] >= race.lim;
        const unsigned long long bal = __ballot(c);
        if (bal == 0ull) continue;  // uniform
        put(c, bal, v[j], base + j);  // < 64 before, < 128 after
        if (qn >= 64) {
          qn -= 64;
          draw(qn + lane);
        }
      }
      write_mask(bits, base);
    });
  }
  if (lane < qn) draw(lane);
}

// Slices, launch 1: each slice's maximum and the best race score of its
// threads' maxima (a bound for the race: every finite token is kept).
template <typename T>
__global__ __launch_bounds__(kSampleThreads) void sample_max_kernel(const T *__restrict__ logits, int64_t row_stride,
                                                                    int vocab, SampleArgs a, Slices sl) {
  __shared__ float redv[kSampleThreads / 64];
  __shared__ int64_t redi[kSampleThreads / 64];
  const int s = blockIdx.x, b = blockIdx.y;
  const Row<T> row(logits, row_stride, vocab, a, b);
  const int64_t lo = static_cast<int64_t>(s) * sl.slice;
  const int64_t hi = lo + sl.slice < vocab ? lo + sl.slice : vocab;
  float tmx = -INFINITY;
  const int tmi = track_max<T>(row, lo, hi, tmx);
  const float m = block_max(tmx, redv);
  const bool finite = order_key(tmx) >= order_key(-3.402823466e38f);
  if (row.greedy) {  // the winner: the maximum, at its lowest index
    int64_t at = finite ? tmi : kNoToken;
    block_argmax(tmx, at, redv, redi);
    if (threadIdx.x == 0) {
      sl.rows[b].vmax[s] = m;
      sl.rows[b].best[s] = tmx;
      sl.rows[b].win[s] = at < vocab ? static_cast<int32_t>(at) : 0x7fffffff;
    }
    return;
  }
  const float sc = block_max(finite ? tmx - log_exp_variate(row_stream(a, b), tmi) : -INFINITY, redv);
  if (threadIdx.x == 0) {
    sl.rows[b].vmax[s] = m;
    sl.rows[b].score[s] = sc;
  }
}

// Slices, launch 2: each slice's part of the final pass.
template <typename T>
__global__ __launch_bounds__(kSampleThreads) void sample_slice_kernel(const T *__restrict__ logits,
                                                                      int64_t row_stride, int vocab, SampleArgs a,
                                                                      Slices sl) {
  __shared__ float redv[kSampleThreads / 64];
  __shared__ int64_t redi[kSampleThreads / 64];
  __shared__ float fq_x[kSampleThreads / 64][kFastQueue];  // draw queues (value, token)
  __shared__ int32_t fq_t[kSampleThreads / 64][kFastQueue];
  const int s = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  SliceRow &sr = sl.rows[b];
  const Row<T> row(logits, row_stride, vocab, a, b);
  const int64_t lo = static_cast<int64_t>(s) * sl.slice;
  const int64_t hi = lo + sl.slice < vocab ? lo + sl.slice : vocab;
  const float mx = wave_max(lane < sl.S ? sr.vmax[lane] : -INFINITY);
  Race race{row.greedy, row_stream(a, b), -INFINITY};
  if (row.greedy) {
    race.bi = 0;  // launch 1 found the winner
  } else {
    // the maximum's least possible score (ln E <= 2.812), or the threads' best; nothing finite: no bound
    const float score = wave_max(lane < sl.S ? sr.score[lane] : -INFINITY);
    race.lim = fmaxf(mx - 2.9f, score) - kScoreReach;
  }
  float z = 0.f;
  int cnt = 0;
  uint32_t *mask_row = a.mask ? a.mask + static_cast<int64_t>(b) * ((vocab + 31) / 32) : nullptr;
  final_pass<T>(row, lo, hi, min_key(0.f, mx), mx, race, &fq_x[tid >> 6][0], &fq_t[tid >> 6][0], mask_row, z, cnt);
  const float zs = block_sum(z, redv);
  const float cs = block_sum(static_cast<float>(cnt), redv);
  if (tid == 0) {
    sr.z[s] = zs;
    sr.cnt[s] = static_cast<int32_t>(cs);
  }
  if (row.greedy) return;
  block_argmax(race.best, race.bi, redv, redi);
  if (tid == 0) {
    sr.best[s] = race.best;
    sr.win[s] = race.bi < vocab ? static_cast<int32_t>(race.bi) : 0x7fffffff;
  }
}

// Slices, launch 3: one wave joins a row's slices.
template <typename T>
__global__ __launch_bounds__(64) void sample_join_kernel(const T *__restrict__ logits, int64_t row_stride, int vocab,
                                                         SampleArgs a, Slices sl) {
  const int b = blockIdx.x, lane = threadIdx.x;
  const SliceRow &sr = sl.rows[b];
  const bool on = lane < sl.S;
  const float mx = wave_max(on ? sr.vmax[lane] : -INFINITY);
  if (!(mx > -INFINITY)) {  // nothing finite: token 0, empty support (the slices wrote an empty mask)
    if (lane == 0) {
      a.tokens[b] = 0;
      if (a.logprobs) a.logprobs[b] = -INFINITY;
      if (a.counts) a.counts[b] = 0;
    }
    return;
  }
  float best = on ? sr.best[lane] : -INFINITY;
  int64_t bi = on ? sr.win[lane] : kNoToken;
  wave_argmax(best, bi);
  const float z = wave_sum(on ? sr.z[lane] : 0.f);
  const int cnt = wave_reduce(on ? sr.cnt[lane] : 0, [](int x, int y) { return x + y; });
  if (lane == 0) {
    const Row<T> row(logits, row_stride, vocab, a, b);
    const bool drawn = bi < vocab;
    a.tokens[b] = drawn ? bi : 0;
    if (a.logprobs) a.logprobs[b] = drawn ? (row.x_of(bi) - mx) - logf(z) : -INFINITY;
    if (a.counts) a.counts[b] = cnt;
  }
}

// A whole row per workgroup.
template <typename T>
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(const T *__restrict__ logits, int64_t row_stride,
                                                                int vocab, SampleArgs a) {
  __shared__ float redv[kSampleThreads / 64];
  __shared__ int64_t redi[kSampleThreads / 64];
  __shared__ unsigned long long hist[256];
  __shared__ uint32_t sel_prefix;
  __shared__ unsigned long long sel_above;
  __shared__ unsigned long long red64[kSampleThreads / 64];
  __shared__ uint32_t fcnt[kBins];             // also the ranked select's counts
  __shared__ unsigned long long fmass[kBins];  // also the groups to read again, and the ranked select's masses
  static_assert(sizeof(fmass) >= kGroups * kSampleThreads * 2, "every group fits the list of groups to read again");
  // the final pass's draw queues, or the list path's mask
  __shared__ uint32_t ubuf[kSampleThreads / 64 * kFastQueue * 2];
  static_assert(kSampleThreads / 64 * kFastQueue * 2 >= kMaskWords, "the mask fits the queues");
  __shared__ float gmax[kGroups][kSampleThreads];  // group maxima
  __shared__ uint32_t ckey[kCand];
  __shared__ float cx[kCand];
  __shared__ int32_t cidx[kCand];
  __shared__ int ncand, sel_bin, nhit;
  __shared__ unsigned long long sel_n;
  const int b = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int words = (vocab + 31) / 32;
  const Row<T> row(logits, row_stride, vocab, a, b);
  const bool greedy = row.greedy;
  auto x8 = [&](float v[kVec], int64_t base) { row.x8(v, base); };
  const int64_t step8 = kStep8;
  auto for_chunks = [&](auto every, auto &&f) __attribute__((always_inline)) {
    row.template for_chunks<batch_chunks<T>()>(every, 0, vocab, f);
  };
  auto for_chunks2 = [&](auto every, auto &&f) __attribute__((always_inline)) {
    row.template for_chunks<2>(every, 0, vocab, f);
  };

  // Pass 1: the row maximum. Each thread keeps its own (top_k's capture range)
  // and, for rows drawn by the full-row pass, where it is (the race's bound),
  // or the maxima of its groups of chunks (which of them hold listed tokens).
  const int topk = a.top_k ? a.top_k[b] : 0;
  const float tp = a.top_p ? a.top_p[b] : 1.f;
  const float mp = a.min_p ? a.min_p[b] : 0.f;
  const bool want_k = topk > 0 && topk < vocab;
  const bool want_p = tp < 1.f;
  const bool want_m = mp > 0.f && !want_k && !want_p;  // min_p alone
  // (a row of one chunk per thread under min_p: the pass is as short as its groups, 2,000
  // tokens 10.5 us against 11.1)
  const bool use_g = (want_m && vocab > kStep8) || (want_k && topk <= kSampleThreads);
  const int gsh = a.group_shift, gmask = (1 << gsh) - 1;
  const bool track = !want_k && !want_p && !use_g;
  float tmx = -INFINITY;
  int tmi = 0;
  float mx;
  {
    if (track) {
      tmi = track_max<T>(row, 0, vocab, tmx);
    } else if (use_g) {
      int c = 0;  // uniform
      float gm = -INFINITY;
      for_chunks(Every{}, [&](const float v[kVec], int64_t) __attribute__((always_inline)) {
        gm = fmaxf(gm, max8(v));
        if ((++c & gmask) == 0) {
          gmax[(c >> gsh) - 1][tid] = gm;
          tmx = fmaxf(tmx, gm);
          gm = -INFINITY;
        }
      });
      if (c & gmask) gmax[c >> gsh][tid] = gm;
      tmx = fmaxf(tmx, gm);
    } else {
      for_chunks(Own{}, [&](const float v[kVec], int64_t) __attribute__((always_inline)) { tmx = fmaxf(tmx, max8(v)); });
    }
    mx = block_max(tmx, redv);
  }
  if (!(mx > -INFINITY)) {  // nothing finite: token 0, empty support
    if (tid == 0) {
      a.tokens[b] = 0;
      if (a.logprobs) a.logprobs[b] = -INFINITY;
      if (a.counts) a.counts[b] = 0;
    }
    if (a.mask)
      for (int wd = tid; wd < words; wd += kSampleThreads) a.mask[static_cast<int64_t>(b) * words + wd] = 0u;
    return;
  }
  uint32_t key_lo = min_key(mp, mx);

  bool fallback = false;
  bool listed = false;  // the LDS list holds every kept token the threshold can keep
  int n = 0;            // its length
  unsigned long long mtot = 0;  // the kept mass of the row (top_p alone)
  bool bin_only = false;        // the list holds the threshold's bin alone, under
  unsigned long long base_cnt = 0, base_mass = 0;  // so many kept tokens and so much (top_p alone) mass
  auto bin_of = [&](float x) {
    const float d = (mx - x) * kBinScale;  // NaN and -inf land in the open bin (and are not kept)
    return d < static_cast<float>(kBins - 1) ? static_cast<int>(d) : kBins - 1;
  };
  // Appends the kept tokens with `take` set to the list (one LDS atomic per
  // wave and slot); every lane of the wave that is still in the pass calls it.
  // `lost` is called for a token the full list has no room for. True
  // (uniform): the list has overflowed.
  auto append_or = [&](bool take, float x, int64_t t, auto &&lost) -> bool {
    const unsigned long long bal = __ballot(take);
    if (bal == 0ull) return false;  // uniform: most slots of most passes
    const int first = __ffsll(static_cast<long long>(bal)) - 1;
    int at = 0;
    if (lane == first) at = atomicAdd(&ncand, __popcll(bal));
    const int at0 = __builtin_amdgcn_readlane(at, first);
    at = at0 + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(bal >> 32),
                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bal), 0u));
    if (take) {
      if (at < kCand) {
        ckey[at] = order_key(x);
        cx[at] = x;
        cidx[at] = static_cast<int32_t>(t);
      } else {
        lost();
      }
    }
    return at0 + __popcll(bal) > kCand;
  };
  auto append = [&](bool take, float x, int64_t t) { (void)append_or(take, x, t, [] {}); };
  if (want_k || want_p || (want_m && use_g)) {
    const bool hmass = want_p && !want_k;  // after top_k, top_p runs on the list
    for (int j = tid; j < kBins; j += kSampleThreads) {
      fcnt[j] = 0u;
      fmass[j] = 0ull;
    }
    if (tid == 0) {
      ncand = 0;
      nhit = 0;
      sel_n = 0ull;
    }
    __syncthreads();

    // Capture range, in bins below the maximum, holding every token the
    // threshold can keep. top_k (k <= threads): the k largest of the threads'
    // maxima are k distinct tokens, so the row's k-th largest lies in or above
    // the bin of their k-th. top_p alone: top_p_bins. min_p: every kept token.
    int bcap = kBins - 1;
    if (want_k && topk <= kSampleThreads) {
      atomicAdd(&fcnt[bin_of(tmx)], 1u);
      __syncthreads();
      const unsigned long long c0 = fcnt[2 * tid], c1 = fcnt[2 * tid + 1];
      unsigned long long ctot;
      const unsigned long long cex = block_exscan_u64(c0 + c1, red64, ctot);
      const unsigned long long kk = static_cast<unsigned long long>(topk);
      if (tid == 0) sel_bin = kBins - 1;
      __syncthreads();
      if (cex < kk && kk <= cex + c0)
        sel_bin = 2 * tid;
      else if (cex + c0 < kk && kk <= cex + c0 + c1)
        sel_bin = 2 * tid + 1;
      fcnt[2 * tid] = 0u;
      fcnt[2 * tid + 1] = 0u;
      __syncthreads();
      bcap = sel_bin;
    } else if (!want_k && !want_m) {
      bcap = top_p_bins(tp, vocab);
    }

    // Capture: the kept tokens within the range go to the list, and those past
    // its end to the threshold's histogram (which takes the list's too if it
    // overflowed); top_p alone also sums the kept mass over the whole row (a
    // token kMassBins or more below the maximum weighs under one fixed-point
    // unit: exactly 0).
    // The bin tests are distance compares: with d = (mx - x) * kBinScale as
    // bin_of forms it (d >= 0: x <= mx; NaN and -inf fail every compare),
    // bin <= bcap <=> d < bcap + 1 and bin < kMassBins <=> d < kMassBins
    // (bcap + 1 <= kBins - 1). The bin is formed only for the few tokens taken.
    // A row with an infinite maximum has no distances (inf - inf is NaN, which no
    // range holds): the key alone decides there, over the whole row.
    const bool captured = mx < INFINITY && (want_m || bcap < kBins - 1);
    const float bcap1 = want_m ? INFINITY : static_cast<float>(bcap + 1);
    if (captured && use_g) {
      // The groups whose maximum is in the range, a lane per chunk.
      uint16_t *hits = reinterpret_cast<uint16_t *>(fmass);  // the top_p mass bins are not used with top_k or min_p
      const int n_g = (((vocab + kStep8 - 1) / kStep8 - 1) >> gsh) + 1;
      for (int g = 0; g < n_g; ++g) {
        const float m = gmax[g][tid];
        const bool hit = order_key(m) >= key_lo && (mx - m) * kBinScale < bcap1;
        const unsigned long long bal = __ballot(hit);
        if (bal == 0ull) continue;  // uniform
        const int first = __ffsll(static_cast<long long>(bal)) - 1;
        int at = 0;
        if (lane == first) at = atomicAdd(&nhit, __popcll(bal));
        at = __shfl(at, first, 64) + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(bal >> 32),
                                                                __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bal), 0u));
        if (hit) hits[at] = static_cast<uint16_t>(g * kSampleThreads + tid);
      }
      __syncthreads();
      const int nh = nhit;
      if (!want_m || nh << gsh <= kMaxHitChunks) {
        for (int t = tid; t < nh << gsh; t += kSampleThreads) {
          const int h = hits[t >> gsh];
          const int64_t base = static_cast<int64_t>((h / kSampleThreads << gsh) + (t & gmask)) * kStep8 +
                               static_cast<int64_t>(h % kSampleThreads) * kVec;
          if (base >= vocab) continue;
          float v[kVec];
          x8(v, base);
#pragma unroll
          for (int j = 0; j < kVec; ++j) {
            const float d = (mx - v[j]) * kBinScale;
            const bool take = order_key(v[j]) >= key_lo && d < bcap1;
            if (take && !want_m) atomicAdd(&fcnt[static_cast<int>(d)], 1u);
            append(take, v[j], base + j);
          }
        }
        __syncthreads();
        n = ncand;
        listed = n > 0 && n <= kCand;
      }
      __syncthreads();
    } else if (captured) {  // top_p alone
      unsigned long long tmass = 0;
      // The key test is one float compare when the threshold is a negative
      // float (NEG; see the fast final loop).
      const float thr = __uint_as_float(~key_lo);  // with NEG: the keep threshold as a float
      // (one instance per key test: a select on it would do both)
      bool over = false;
      auto capture = [&](auto neg) __attribute__((always_inline)) {
        constexpr bool NEG = decltype(neg)::value;
        for_chunks2(Own{}, [&](const float v[kVec], int64_t base) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < kVec; ++j) {
            const float d = (mx - v[j]) * kBinScale;
            const bool kept = NEG ? v[j] >= thr : order_key(v[j]) >= key_lo;
            unsigned long long m = 0;
            if (kept && d < static_cast<float>(kMassBins)) m = fixed_mass(v[j], mx);
            tmass += m;
            const bool take = kept && d < bcap1;
            auto count = [&] {
              const int bn = static_cast<int>(d);
              atomicAdd(&fcnt[bn], 1u);
              atomicAdd(&fmass[bn], m);
            };
            if (!over)
              over = append_or(take, v[j], base + j, count);
            else if (take)
              count();
          }
        });
      };
      if (key_lo < 0x80000000u)
        capture(std::true_type{});
      else
        capture(std::false_type{});
      const unsigned long long wm = wave_sum_u64(tmass);
      if (lane == 0) atomicAdd(&sel_n, wm);
      __syncthreads();
      n = ncand;
      listed = n > 0 && n <= kCand;
      mtot = sel_n;
      if (!listed) {  // the list's own tokens join the histogram
        for (int i = tid; i < kCand; i += kSampleThreads) {
          const int bn = static_cast<int>((mx - cx[i]) * kBinScale);
          atomicAdd(&fcnt[bn], 1u);
          if (hmass) atomicAdd(&fmass[bn], fixed_mass(cx[i], mx));
        }
      }
      __syncthreads();
    }

    if (!listed && !want_m) {
      // The threshold's bin from the histogram -- the capture's, which holds
      // the threshold, or one pass over the whole row -- then a compaction
      // pass: every kept token at or above that bin.
      if (tid == 0) ncand = 0;
      if (!captured) {
        uint32_t tcnt = 0;
        unsigned long long tmass = 0;  // this thread's share of the open bin
        for_chunks2(Own{}, [&](const float v[kVec], int64_t) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < kVec; ++j) {
            if (order_key(v[j]) < key_lo) continue;
            const int bn = bin_of(v[j]);
            const unsigned long long m = hmass ? fixed_mass(v[j], mx) : 0ull;
            if (bn == kBins - 1) {
              ++tcnt;
              tmass += m;
            } else {
              atomicAdd(&fcnt[bn], 1u);
              if (hmass) atomicAdd(&fmass[bn], m);
            }
          }
        });
        const unsigned long long wc = wave_sum_u64(tcnt), wm = wave_sum_u64(tmass);
        if (lane == 0) {
          atomicAdd(&fcnt[kBins - 1], static_cast<uint32_t>(wc));
          if (hmass) atomicAdd(&fmass[kBins - 1], wm);
        }
      }
      __syncthreads();
      // Threshold bin from scans over the bins in value order (bin 0 = nearest the max).
      const unsigned long long c0 = fcnt[2 * tid], c1 = fcnt[2 * tid + 1];
      unsigned long long ctot;
      const unsigned long long cex = block_exscan_u64(c0 + c1, red64, ctot);
      unsigned long long m0 = 0, m1 = 0, mex = 0;
      if (hmass) {
        m0 = fmass[2 * tid];
        m1 = fmass[2 * tid + 1];
        unsigned long long htot;
        mex = block_exscan_u64(m0 + m1, red64, htot);
        if (!captured) mtot = htot;  // else the capture pass summed the whole row
      }
      if (tid == 0) sel_bin = -1;
      __syncthreads();
      if (want_k) {
        const unsigned long long kk = static_cast<unsigned long long>(topk);
        if (ctot >= kk) {  // else fewer than k kept tokens: the full-row path keeps them all
          if (cex < kk && kk <= cex + c0) {
            sel_bin = 2 * tid;
            sel_n = cex + c0;
          } else if (cex + c0 < kk && kk <= cex + c0 + c1) {
            sel_bin = 2 * tid + 1;
            sel_n = cex + c0 + c1;
          }
        }
      } else {
        const unsigned long long target = top_p_target(tp, mtot);
        if (mex < target && target <= mex + m0) {
          sel_bin = 2 * tid;
          sel_n = cex + c0;
        } else if (mex + m0 < target && target <= mex + m0 + m1) {
          sel_bin = 2 * tid + 1;
          sel_n = cex + c0 + c1;
        }
      }
      __syncthreads();
      const int tb = sel_bin;
      const unsigned long long n_list = sel_n;
      // More tokens above the threshold's bin than the list holds: the list
      // takes that bin alone, and the select counts from what lies above it.
      const unsigned long long n_bin = tb >= 0 ? fcnt[tb] : 0u;
      bin_only = n_list > static_cast<unsigned long long>(kCand);
      fallback = tb < 0 || tb == kBins - 1 || (bin_only && n_bin > static_cast<unsigned long long>(kCand));
      if (!fallback && bin_only) {
        __syncthreads();  // everyone has read sel_n
        if (tid == (tb >> 1)) {
          sel_n = n_list - n_bin;
          sel_above = (tb & 1) ? mex + m0 : mex;
        }
        __syncthreads();
        base_cnt = sel_n;
        base_mass = sel_above;
        for_chunks(Own{}, [&](const float v[kVec], int64_t base) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < kVec; ++j) append(order_key(v[j]) >= key_lo && bin_of(v[j]) == tb, v[j], base + j);
        });
        __syncthreads();
        n = ncand;  // == n_bin
        listed = true;
      } else if (!fallback) {
        for_chunks(Own{}, [&](const float v[kVec], int64_t base) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < kVec; ++j) append(order_key(v[j]) >= key_lo && bin_of(v[j]) <= tb, v[j], base + j);
        });
        __syncthreads();
        n = ncand < kCand ? ncand : kCand;  // == n_list
        listed = true;
      }
    }

    if (listed && n <= (want_k && want_p ? kRanked : kRankedOne) && !want_m) {
      // Ranked select: every entry counts the entries above it and their mass
      // (the threads share each entry's n compares), then top_k keeps an entry
      // iff fewer than k are above it (ties kept) and top_p iff the kept mass
      // above it is short of the target. Five barriers; the radix select below
      // takes 16 per threshold (about 5 us each), but n^2 compares outlast it.
      int np = 64;
      while (np < n) np <<= 1;
      const int i = tid & (np - 1), parts = kSampleThreads / np, part = tid / np;
      if (want_p && tid < n) fmass[tid] = fixed_mass(cx[tid], mx);
      fcnt[tid] = 0u;
      fmass[kSampleThreads + tid] = 0ull;
      __syncthreads();
      const uint32_t key = i < n ? ckey[i] : 0xffffffffu;
      uint32_t above = 0;
      unsigned long long mass = 0;
      for (int j = part; j < n; j += parts) {
        const bool g = ckey[j] > key;
        above += g ? 1u : 0u;
        if (want_p) mass += g ? fmass[j] : 0ull;
      }
      if (above != 0u) atomicAdd(&fcnt[i], above);
      if (mass != 0ull) atomicAdd(&fmass[kSampleThreads + i], mass);
      if (tid == 0) sel_prefix = 0xffffffffu;
      __syncthreads();
      bool keep = tid < n && (!want_k || fcnt[tid] + base_cnt < static_cast<unsigned long long>(topk));
      if (want_p && !(want_k && bin_only)) {
        // After top_k the list holds every kept token, so the kept mass sums
        // over it; top_p alone keeps the whole row's mass.
        unsigned long long total = mtot;
        if (want_k) (void)block_exscan_u64(keep ? fmass[tid] : 0ull, red64, total);
        keep = keep && base_mass + fmass[kSampleThreads + tid] < top_p_target(tp, total);
      }
      if (keep) atomicMin(&sel_prefix, ckey[tid]);
      __syncthreads();
      const uint32_t least = sel_prefix;
      if (least != 0xffffffffu && least > key_lo) key_lo = least;
      __syncthreads();
    } else if (listed && !want_m) {
      // top_k on the list: the k-th largest key (ties kept). Every list entry
      // is kept; a list shorter than k holds every kept token, all of which stay.
      if (want_k && base_cnt + n >= static_cast<unsigned long long>(topk)) {
        uint32_t prefix = 0, pmask = 0;
        unsigned long long remaining = static_cast<unsigned long long>(topk) - base_cnt;
        for (int shift = 24; shift >= 0; shift -= 8) {
          for (int j = tid; j < 256; j += kSampleThreads) hist[j] = 0ull;
          __syncthreads();
          for (int i = tid; i < n; i += kSampleThreads) {
            const uint32_t k = ckey[i];
            if ((k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1ull);
          }
          __syncthreads();
          find_from_top(hist, 0ull, remaining, &sel_prefix, &sel_above);  // found: the list holds >= k keys
          __syncthreads();
          remaining -= sel_above;
          prefix |= sel_prefix << shift;
          pmask |= 255u << shift;
          __syncthreads();
        }
        if (prefix > key_lo) key_lo = prefix;
      }
      // top_p on the list. After top_k the list holds every kept token (its
      // keys >= key_lo), so the kept mass sums over it; top_p alone keeps the
      // whole row's mass.
      if (want_p && !(want_k && bin_only)) {
        unsigned long long total = mtot;
        if (want_k) {
          unsigned long long part = 0;
          for (int i = tid; i < n; i += kSampleThreads)
            if (ckey[i] >= key_lo) part += fixed_mass(cx[i], mx);
          (void)block_exscan_u64(part, red64, total);
        }
        const unsigned long long target = top_p_target(tp, total);
        uint32_t prefix = 0, pmask = 0;
        unsigned long long above = base_mass;
        for (int shift = 24; shift >= 0; shift -= 8) {
          for (int j = tid; j < 256; j += kSampleThreads) hist[j] = 0ull;
          __syncthreads();
          for (int i = tid; i < n; i += kSampleThreads) {
            const uint32_t k = ckey[i];
            if (k >= key_lo && (k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], fixed_mass(cx[i], mx));
          }
          __syncthreads();
          find_from_top(hist, above, target, &sel_prefix, &sel_above);
          __syncthreads();
          prefix |= sel_prefix << shift;
          above = sel_above;
          pmask |= 255u << shift;
          __syncthreads();
        }
        if (prefix > key_lo) key_lo = prefix;
      }
    }
    if (bin_only) listed = false;  // the final pass takes the row
  }

  // top_k over the whole row: radix select of the k-th largest kept key.
  if (fallback && want_k) {
    uint32_t prefix = 0, pmask = 0;
    unsigned long long remaining = static_cast<unsigned long long>(topk);
    bool enough = true;
    for (int shift = 24; shift >= 0; shift -= 8) {
      for (int j = tid; j < 256; j += kSampleThreads) hist[j] = 0ull;
      __syncthreads();
      for (int64_t base = static_cast<int64_t>(tid) * kVec; base < vocab; base += step8) {
        float v[kVec];
        x8(v, base);
#pragma unroll
        for (int j = 0; j < kVec; ++j) {
          const uint32_t k = order_key(v[j]);
          if (k >= key_lo && (k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1ull);
        }
      }
      __syncthreads();
      find_from_top(hist, 0ull, remaining, &sel_prefix, &sel_above);  // -1: fewer than k kept tokens
      __syncthreads();
      const int bin = static_cast<int>(sel_prefix);
      const unsigned long long above = sel_above;
      __syncthreads();
      if (bin < 0) {
        enough = false;
        break;
      }
      remaining -= above;
      prefix |= static_cast<uint32_t>(bin) << shift;
      pmask |= 255u << shift;
    }
    if (enough && prefix > key_lo) key_lo = prefix;
  }

  // top_p over the whole row: radix select over fixed-point mass
  // w_i = exp(x_i - max) * 2^32.
  if ((fallback || (bin_only && want_k)) && want_p) {
    unsigned long long total = 0;
    {
      // total kept mass (integer: exact, order-independent)
      for (int j = tid; j < 256; j += kSampleThreads) hist[j] = 0ull;
      __syncthreads();
      unsigned long long part = 0;
      for (int64_t base = static_cast<int64_t>(tid) * kVec; base < vocab; base += step8) {
        float v[kVec];
        x8(v, base);
#pragma unroll
        for (int j = 0; j < kVec; ++j)
          if (order_key(v[j]) >= key_lo) part += fixed_mass(v[j], mx);
      }
      atomicAdd(&hist[0], part);
      __syncthreads();
      total = hist[0];
      __syncthreads();
    }
    const unsigned long long target = top_p_target(tp, total);
    uint32_t prefix = 0, pmask = 0;
    unsigned long long above = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
      for (int j = tid; j < 256; j += kSampleThreads) hist[j] = 0ull;
      __syncthreads();
      for (int64_t base = static_cast<int64_t>(tid) * kVec; base < vocab; base += step8) {
        float v[kVec];
        x8(v, base);
#pragma unroll
        for (int j = 0; j < kVec; ++j) {
          const uint32_t k = order_key(v[j]);
          if (k >= key_lo && (k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], fixed_mass(v[j], mx));
        }
      }
      __syncthreads();
      find_from_top(hist, above, target, &sel_prefix, &sel_above);  // target <= total: always found
      __syncthreads();
      prefix |= sel_prefix << shift;
      above = sel_above;
      pmask |= 255u << shift;
      __syncthreads();
    }
    if (prefix > key_lo) key_lo = prefix;
  }

  Race race{greedy, row_stream(a, b), -INFINITY};
  int cnt = 0;
  float lz;  // ln of the kept mass, in units of the maximum's weight
  // The race's bound starts from the maximum's least possible score (ln E <=
  // 2.812; the maximum is always kept), or from the best score of the threads'
  // kept maxima where pass 1 kept them.
  if (!greedy) {
    race.lim = mx - 2.9f;
    if (track) {
      const float s0 = order_key(tmx) >= key_lo ? tmx - log_exp_variate(race.stream, tmi) : -INFINITY;
      race.lim = fmaxf(race.lim, block_max(s0, redv));
    }
    race.lim -= kScoreReach;
  } else if (track && tmx == mx) {  // a greedy row's winner: the maximum, at its lowest index
    race.best = tmx;
    race.bi = tmi;
  } else if (track) {
    race.bi = kNoToken - 1;  // another thread has it
  }
  if (listed) {
    // Final step on the list, which holds every kept token: the kept mass in
    // fixed point (exact, so independent of the list's order), the draw, the
    // mask (assembled in LDS) and the support size.
    uint32_t *mbits = ubuf;
    const int nw0 = words < kMaskWords ? words : kMaskWords;
    if (a.mask)
      for (int wd = tid; wd < nw0; wd += kSampleThreads) mbits[wd] = 0u;
    __syncthreads();
    unsigned long long zf = 0;
    for (int i = tid; i < n; i += kSampleThreads) {
      if (ckey[i] < key_lo) continue;
      const float x = cx[i];
      const int64_t t = cidx[i];
      zf += fixed_mass(x, mx);
      ++cnt;
      race.run(x, t);
      if (a.mask && (t >> 5) < nw0) atomicOr(&mbits[t >> 5], 1u << (t & 31));
    }
    unsigned long long ztot;
    (void)block_exscan_u64(zf, red64, ztot);  // its barriers also complete the mask
    lz = static_cast<float>(log(static_cast<double>(ztot)) - 22.180709777918249);  // - ln 2^32
    if (a.mask)
      for (int wd = tid; wd < nw0; wd += kSampleThreads) a.mask[static_cast<int64_t>(b) * words + wd] = mbits[wd];
    if (a.mask && words > kMaskWords) {  // uniform: the mask's further words, kMaskWords at a time
      for (int w0 = kMaskWords; w0 < words; w0 += kMaskWords) {
        __syncthreads();
        const int nw = words - w0 < kMaskWords ? words - w0 : kMaskWords;
        for (int wd = tid; wd < nw; wd += kSampleThreads) mbits[wd] = 0u;
        __syncthreads();
        for (int i = tid; i < n; i += kSampleThreads) {
          const int wd = (cidx[i] >> 5) - w0;
          if (ckey[i] >= key_lo && wd >= 0 && wd < nw) atomicOr(&mbits[wd], 1u << (cidx[i] & 31));
        }
        __syncthreads();
        for (int wd = tid; wd < nw; wd += kSampleThreads) a.mask[static_cast<int64_t>(b) * words + w0 + wd] = mbits[wd];
      }
    }
  } else {
    float z = 0.f;
    float *qx = reinterpret_cast<float *>(ubuf) + (tid >> 6) * kFastQueue;
    int32_t *qt = reinterpret_cast<int32_t *>(ubuf) + (kSampleThreads / 64 + (tid >> 6)) * kFastQueue;
    uint32_t *mask_row = a.mask ? a.mask + static_cast<int64_t>(b) * words : nullptr;
    final_pass<T>(row, 0, vocab, key_lo, mx, race, qx, qt, mask_row, z, cnt);
    lz = logf(block_sum(z, redv));
  }
  block_argmax(race.best, race.bi, redv, redi);
  const float c = block_sum(static_cast<float>(cnt), redv);
  if (tid == 0) {
    const bool drawn = race.bi < vocab;  // (the maximum is always kept; no index past the row is ever read)
    a.tokens[b] = drawn ? race.bi : 0;
    if (a.logprobs) a.logprobs[b] = drawn ? (row.x_of(race.bi) - mx) - lz : -INFINITY;
    if (a.counts) a.counts[b] = static_cast<int32_t>(c);
  }
}

// Slices of a launch over `batch` rows drawn from the whole vocabulary: about
// one workgroup per CU in the two sliced launches. 1: whole rows. Measured (us
// per call, sliced against whole rows): 151,936 tokens 1 row 20 / 47, 32 rows
// 28 / 74, 128 rows 61 / 79; 50,000 tokens 1 row 20 / 21, 64 rows 25 / 32, 96
// rows 35 / 33; 32,001 tokens 1 row 21 / 18. (Rows under top_k or min_p read
// little of the row twice and stay whole: 21 us and 15 us at 151,936 tokens.)
static Slices sample_slices(int batch, int vocab) {
  Slices s{nullptr, 1, 0};
  const int chunks = (vocab + kStep8 - 1) / kStep8;
  if (batch <= 0 || batch > kSliceRows) return s;
  int per = (chunks * batch + 255) / 256;  // chunks per slice
  const int least = (chunks + kMaxSlices - 1) / kMaxSlices;
  per = per < least ? least : per;
  if (chunks - per < kMinSliceGain) return s;
  s.S = (chunks + per - 1) / per;
  s.slice = per * kStep8;
  return s;
}

// kGroupShift up to 262,144 tokens, one more for every doubling.
static int sample_group_shift(int vocab) {
  int s = kGroupShift;
  while ((static_cast<int64_t>(kGroups) << s) * kStep8 < vocab) ++s;
  return s;
}

}  // namespace wkv

using namespace wkv;

static int launch_sample(const void *logits, int32_t logits_dtype, int64_t row_stride, int32_t batch, int32_t vocab,
                         const SampleArgs &a, void *workspace, int64_t workspace_bytes, void *stream) {
  WKV_CHECK_ARG(batch >= 0, "batch must be >= 0");
  if (batch == 0) return WKV_OK;
  WKV_CHECK_ARG(vocab > 0 && vocab < (1 << 24), "vocab must be in [1, 2^24) (got %d)", vocab);
  WKV_CHECK_ARG(logits != nullptr && a.tokens != nullptr, "logits / out_tokens is NULL");
  WKV_CHECK_ARG(logits_dtype == 0 || logits_dtype == 1, "logits_dtype must be 0 (fp32) or 1 (bf16)");
  WKV_CHECK_ARG(row_stride >= vocab, "row_stride %lld < vocab %d", (long long)row_stride, vocab);
  auto s = static_cast<hipStream_t>(stream);
  Slices sl{nullptr, 1, 0};
  if (workspace != nullptr && a.top_k == nullptr && a.top_p == nullptr && a.min_p == nullptr) {
    sl = sample_slices(batch, vocab);
    sl.rows = static_cast<SliceRow *>(workspace);
    const int64_t need = static_cast<int64_t>(batch) * static_cast<int64_t>(sizeof(SliceRow));
    if (sl.S > 1)
      WKV_CHECK_ARG(aligned16(workspace) && workspace_bytes >= need, "workspace too small: need %lld bytes, got %lld",
                    (long long)need, (long long)workspace_bytes);
  }
  const dim3 grid(static_cast<unsigned>(sl.S), static_cast<unsigned>(batch));
#define WKV_SAMPLE(Tv)                                                                                          \
  do {                                                                                                          \
    auto p = static_cast<const Tv *>(logits);                                                                   \
    if (sl.S > 1) {                                                                                             \
      sample_max_kernel<Tv><<<grid, kSampleThreads, 0, s>>>(p, row_stride, vocab, a, sl);                       \
      WKV_CHECK_LAUNCH("sample maxima");                                                                        \
      sample_slice_kernel<Tv><<<grid, kSampleThreads, 0, s>>>(p, row_stride, vocab, a, sl);                     \
      WKV_CHECK_LAUNCH("sample slices");                                                                        \
      sample_join_kernel<Tv><<<batch, 64, 0, s>>>(p, row_stride, vocab, a, sl);                                 \
    } else {                                                                                                    \
      sample_kernel<Tv><<<batch, kSampleThreads, 0, s>>>(p, row_stride, vocab, a);                              \
    }                                                                                                           \
  } while (0)
  if (logits_dtype == 0)
    WKV_SAMPLE(float);
  else
    WKV_SAMPLE(uint16_t);
#undef WKV_SAMPLE
  WKV_CHECK_LAUNCH("sample");
  return WKV_OK;
}

extern "C" int64_t wkv_sample_workspace_size(int32_t batch, int32_t vocab) {
  if (batch < 0 || vocab <= 0 || vocab >= (1 << 24)) return -1;
  return sample_slices(batch, vocab).S > 1 ? static_cast<int64_t>(batch) * static_cast<int64_t>(sizeof(SliceRow)) : 0;
}

extern "C" int wkv_sample(const void *logits, int32_t logits_dtype, int64_t row_stride, int32_t batch, int32_t vocab,
                          const float *temperature, const int32_t *top_k, const float *top_p, const float *min_p,
                          const float *repetition_penalty, const uint32_t *seen_tokens, const uint64_t *seeds,
                          int64_t step, int64_t *out_tokens, float *out_logprobs, uint32_t *out_mask,
                          int32_t *out_counts, void *stream) {
  const SampleArgs a{temperature, top_k, top_p, min_p, repetition_penalty, seen_tokens, seeds, step,
                     out_tokens, out_logprobs, out_mask, out_counts, sample_group_shift(vocab)};
  return launch_sample(logits, logits_dtype, row_stride, batch, vocab, a, nullptr, 0, stream);
}

extern "C" int wkv_sample_sliced(const void *logits, int32_t logits_dtype, int64_t row_stride, int32_t batch,
                                 int32_t vocab, const float *temperature, const int32_t *top_k, const float *top_p,
                                 const float *min_p, const float *repetition_penalty, const uint32_t *seen_tokens,
                                 const uint64_t *seeds, int64_t step, int64_t *out_tokens, float *out_logprobs,
                                 uint32_t *out_mask, int32_t *out_counts, void *workspace, int64_t workspace_bytes,
                                 void *stream) {
  const SampleArgs a{temperature, top_k, top_p, min_p, repetition_penalty, seen_tokens, seeds, step,
                     out_tokens, out_logprobs, out_mask, out_counts, sample_group_shift(vocab)};
  return launch_sample(logits, logits_dtype, row_stride, batch, vocab, a, workspace, workspace_bytes, stream);
}
