// GQA prefill / chunked-prefill attention over the paged cache (gfx950).
//
// Sequence b brings qlen_b = cu_seqlens_q[b+1] - cu_seqlens_q[b] new tokens
// at positions [L_b - qlen_b, L_b) (L_b = seq_lens[b]: cached context plus the
// new tokens, which the entry point appends to the cache first). New token j
// attends causally to positions [0, L_b - qlen_b + j] -- the bottom-right
// aligned mask of a varlen prefill over a paged context (a prefix-cache hit or
// an earlier chunk).
//
// Work decomposition: the query rows of one (sequence, KV head) are units of
// one query head x 32 consecutive query tokens, unit u = tile u / G of head
// u % G; a workgroup of four waves takes four consecutive units, one per wave,
// so the MFMA columns are consecutive query tokens of one head and the four
// waves stream the same key tiles. Units run over head and tile together, so
// no wave idles when G is not a multiple of four (G = 7: 7/8 of the waves
// worked when a workgroup held four heads of one tile; G = 2: half of them).
// Every unit group of a (sequence, KV head) re-reads that head's keys, so the
// 1-D grid sends them to one XCD (the dispatcher deals workgroup i to XCD
// i mod 8): the keys are served from that XCD's L2 instead of being fetched by
// all eight. The latest (most expensive, causally) query tiles are dispatched
// first. Keys are copied once per workgroup into LDS by LDS-DMA, in 16-token
// tiles, four per step of 64 keys; each wave holds 32 queries and runs
// 32x32x16 bf16 MFMAs. fp8 tiles are dequantized in LDS (exactly:
// power-of-two scales) by the wave that copied them, so both dtypes share the
// attention arithmetic. Tiles on the causal diagonal mask per lane (column).
// A grid too small for the chip (a few new tokens over a long context) may share
// its 64-key steps evenly over a number of workgroups instead (share_workgroups):
// a workgroup's share may end inside a unit group, whose parts leave fp32
// partials that prefill_merge_kernel combines by log-sum-exp.
#include "gqa_tiles.h"
#include "lds_dma.h"

#include <cmath>

namespace wkv {

constexpr int kPrefillWaves = 4;
constexpr int kPrefillCus = 256;
constexpr int kShareMinKeys = 1024;  // below, no estimate favours sharing (its second launch alone costs the gain)

// The rule that shares a launch's steps over a number of workgroups compares
// estimates in microseconds, fitted to launches of 8 to 1,000 unit groups over
// 400 to 17,000 keys.
struct ShareCost {
  float alone;  // one 64-key step of a workgroup alone on its CU
  float pair;   // ... of each of two on a CU
  float tail;   // the last workgroups of more than one per CU, as a share of the longest chain
  float gain;   // shared where the estimate is below this share of the plain launch's
};
template <int D, bool FP8>
__host__ __device__ constexpr ShareCost share_cost() {
  return FP8 && D == 64 ? ShareCost{1.2f, 1.5f, 0.1f, 0.85f} : ShareCost{FP8 ? 1.45f : 1.08f, 2.0f, 0.3f, 0.75f};
}
constexpr float kPartUs = 0.05f;   // writing and merging a workgroup's partials
constexpr float kGroupUs = 6.0f;   // starting a unit group (its queries, table and first keys)
constexpr float kLaunchUs = 5.0f;  // a plain launch's fixed part
constexpr float kShareUs = 9.5f;   // a shared launch's: with the prefix and the merge's launch

// Workgroups (a multiple of 64, at most `most`) that are expected to share T
// steps of `groups` unit groups, the longest of `longest` steps, faster than a
// workgroup per group would take them; 0: none. PAID: the shared launch's fixed
// part is spent either way.
// Measured (us, plain -> shared): 4 x 37-250 new tokens over 5-15K keys at
// 28/4 heads 241 -> 131 (fp8 352 -> 131), 64 over 2K at 32/8 38 -> 23,
// 8 x 20-60 over 4-12K at 32/4 fp8 275 -> 82, 1,000 over 8K at 16/8 147 ->
// 87; but 16 x 16 over 1K 22.5 -> 27.3, one prompt of 1,500 tokens 36 -> 55
// and of 512 15 -> 29, two of 2,048 at 14/2 fp8 41 -> 62: short chains gain less
// than the partials and the second launch cost. Over 2,172 shapes (those heads,
// 1-16 sequences, 1-2,048 new tokens over 0-15K) the choice is at worst 11%
// slower than the plain launch (3 by more than 5%) and 4% from the best of both.
template <int D, bool FP8, bool PAID>
__host__ __device__ __forceinline__ int share_workgroups(float T, float longest, float groups, int most) {
  constexpr ShareCost c = share_cost<D, FP8>();
  float best = longest * c.alone;
  if (groups > kPrefillCus) best = fmaxf(best, T / (2 * kPrefillCus) * c.pair) + c.tail * longest * c.alone;
  best = PAID ? best + kShareUs : (best + kLaunchUs) * c.gain;
  int W = 0;
#pragma unroll
  for (int w = 64; w <= 2 * kPrefillCus; w += 64) {
    const bool two = w > kPrefillCus;
    const float us = T * ((two ? c.pair : c.alone) / w) + kPartUs * w * D / 128 +
                     (two ? 0.5f : 1.f) * kGroupUs * (1.f + groups * (1.f / w)) + kShareUs;
    if (w <= most && us < best) {
      best = us;
      W = w;
    }
  }
  return W;
}

// Eight e4m3fn codes (bytes of lo, then hi) times a power-of-two scale as
// eight bf16 values, by the hardware pair conversion (exact: every such
// product is a bf16 value).
__device__ __forceinline__ u32x4 fp8x8_to_bf16_words(uint32_t lo, uint32_t hi, float sc) {
  return u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, sc, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, sc, true)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, sc, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, sc, true))};
}

// One 16-token key tile of one (block, KV head) in LDS, as the MFMAs read it
// (bf16; fp8 tiles are dequantized into the same layout): K as a bf16 cache
// holds it, [D/8 chunks][16 tokens][16 bytes]; V as [2 token octets][D rows]
// [8 tokens] (16-byte pieces, so a copy still moves whole pieces). A lane's
// MFMA operand is one 16-byte LDS read: 16 bytes of one token's K chunk, or
// the 8 tokens of one octet of one V row.
template <int D>
struct LdsTile {
  static constexpr int KB = D * 16 * 2;  // K bytes
  static constexpr int VB = D * 16 * 2;  // V bytes
};

// ---------------------------------------------------------------------------
// 32 queries per wave on 32x32x16 MFMAs, 64 keys per step (four 16-token
// tiles, one copied by each wave). Lane l holds query l % 32 in both
// accumulators. Per step and wave:
//   S^T for keys 0..31 and 32..63 of the step    two chains of D/16 MFMAs
//                                                 32x32x16 (one per half,
//                                                 interleaved: a chain never
//                                                 waits on itself)
//   one row maximum, one rescale test            over the 64 keys
//   P V^T                                        4 x D/32 MFMAs 32x32x16
//   copies of the wave's tile: V of the next     one buffer resource each,
//   step, K of the step after                    16-byte copies (the K copies
//                                                 under one M0)
// so the per-step costs (barriers, waits, loop and mask tests, the maximum's
// cross-lane swap) and the per-tile block lookup fall on 32 MFMAs. Row i of
// each half's S^T carries key kperm(i) of the half (rows 4..7 and 8..11 of
// each 16 swapped), so score r of lane l is key 16 (r/8) + 8 (l/32) + r % 8
// of the half -- the PV B operand as it stands -- and the row sum is taken
// on the packed bf16 probabilities the PV products consume (v_dot2c_f32_bf16
// against 1.0, two per instruction). A block id outside [0, num_blocks) reads block 0: no
// access leaves the cache, and that sequence's output is unspecified.
//
// Software pipeline, one workgroup barrier per step: while a wave finishes
// step s (its probabilities, then its PV products) it scores step s + 1, so
// its MFMAs and its softmax VALU work overlap inside the wave --
//   phase A: the QK products of step s + 1  ||  exponentials, packing and row
//            sum of step s
//   phase B: the PV products of step s      ||  mask, exponents against the
//            reference and their maximum of step s + 1 (the rare move of the
//            reference maximum rescales after the PV products)
// (interleaved by sched_group_barrier: an MFMA, then a few VALU, with the LDS
// operand reads four MFMAs ahead). The copies of a step are one step ahead:
// at the barrier of step s every wave's V of step s and K of step s + 1 have
// landed and every wave is done with step s - 1, whose slots take V of step
// s + 1 and K of step s + 2. LDS (bf16 tiles): K and V in two step slots
// each, 64 KB at d=128, two workgroups per CU at up to 256 VGPRs per wave.
// fp8 caches: the copies land in a staging area of the copying wave's own,
// and that wave dequantizes its tiles into the bf16 layout above with the
// hardware conversion at the (block, head) scale (a power of two: exact in
// bf16) after the wait and before the barrier of the step: its V tile of
// step s and its K tile of step s + 1. The attention arithmetic is the bf16
// one. LDS: 64 KB bf16 plus 8 + 8 KB staging at d=128.
// Division of a non-negative int by a divisor known on the host, in a handful
// of scalar instructions (a runtime division takes some 40 vector ones, and
// half a dozen of them stood in a row before a workgroup's first load: a
// 60-token prompt's launch 8.5 us, 8.0 without them). m = min(floor(2^32 / d), 2^32 - 1) gives a quotient at
// most one too small for every x below 2^31.
struct FastDiv {
  uint32_t m;
  int d;
};

static FastDiv fast_div(int d) {
  return FastDiv{d == 1 ? 0xffffffffu : static_cast<uint32_t>((1ull << 32) / static_cast<uint32_t>(d)), d};
}

__device__ __forceinline__ int operator/(int x, const FastDiv &f) {
  const int q = static_cast<int>(__umulhi(static_cast<uint32_t>(x), f.m));
  return q + (x - q * f.d >= f.d ? 1 : 0);
}

// How a launch covers its work (prefill_grid, on the host).
struct PrefillGrid {
  int n_ug;     // unit groups (four units) per (sequence, KV head), at the longest query
  int R;        // XCDs the unit groups of one (sequence, KV head) are dealt over
  int n_inner;  // workgroups of one (sequence, KV head) per XCD
  int mixed;    // an XCD takes its sub-items' workgroups in turn (by_inner: its sub-items), else one sub-item's after another's
  int n_sub;    // (sequence, KV head) x R
  int W;        // most workgroups that share the steps evenly (share_workgroups); 0: a workgroup per unit group
  int forced;   // the caller's number of them: W whatever the lengths
  int batch;
  int log2R;
  int G;                                  // query heads per KV head
  FastDiv by_U, by_ug, by_inner, by_Hkv;  // units per query tile (G, or more: prefill_grid), n_ug, n_inner, KV heads
};

// The units and 64-key steps of unit group ug of a sequence (uniform).
struct PrefillRange {
  int units;    // units per tile x query tiles of 32 of the sequence
  int kend;     // keys [0, kend) of the group's last query
  int n_steps;  // 64-key steps over them
};

__device__ __forceinline__ PrefillRange prefill_range(int qlen, int L, const FastDiv &U, int ug) {
  PrefillRange r;
  r.units = qlen > 0 ? ((qlen + 31) >> 5) * U.d : 0;
  int u_last = 4 * ug + 3;
  u_last = u_last < r.units ? u_last : r.units - 1;
  const int t_last = u_last >= 0 ? 32 * (u_last / U) : 0;
  const int last = (t_last + 32 < qlen ? t_last + 32 : qlen) - 1;
  r.kend = L - qlen + last + 1;
  r.n_steps = r.kend > 0 ? (r.kend + 63) >> 6 : 0;
  return r;
}

// Shared launches. The steps of every unit group in the order (KV head,
// sequence, unit group) form one line of T steps (a group without keys counts
// one: its rows are written all the same), and workgroup w takes steps
// [w T / W, (w + 1) T / W): every workgroup works equally long whatever the
// mix of lengths, and at most its first and last unit groups are partial.
// pfx[i] (LDS) is the line's prefix at entry i = sequence * n_ug + group of
// one KV head, entries in order, pfx[E] their total; every workgroup forms it
// itself from the lengths (a launch of its own would cost more). The host knows
// bounds of the lengths only: the number of workgroups is chosen here again from
// the lengths themselves, and where sharing does not pay a workgroup takes a
// whole unit group (with bounds of 16,384 keys over prompts of 200 at 32/8 heads, for
// one, that is the plain launch's work with the prefix and an empty merge).
constexpr int kPrefillEntries = 1024;  // at most this many entries per KV head

struct PrefillLine {
  int total, longest, groups;  // of one KV head: steps, steps of the longest unit group, unit groups with queries
};

template <bool STATS>  // else the total alone
__device__ __forceinline__ PrefillLine prefill_prefix(int *pfx, int *red, const int32_t *cu_q,
                                                      const int32_t *seq_lens, int max_seq,
                                                      const PrefillGrid &pg) {
  const int E = pg.batch * pg.n_ug;
  const int per = (E + 64 * kPrefillWaves - 1) / (64 * kPrefillWaves);  // <= 4 entries per thread
  const int e0 = threadIdx.x * per;
  int c[kPrefillEntries / (64 * kPrefillWaves)], sum = 0, mx = 0, n = 0;
#pragma unroll
  for (int k = 0; k < kPrefillEntries / (64 * kPrefillWaves); ++k) {
    c[k] = 0;
    const int e = e0 + k;
    if (k < per && e < E) {
      const int b = e / pg.by_ug, ug = e - b * pg.n_ug;
      const int qlen = cu_q[b + 1] - cu_q[b];
      int L = seq_lens[b];
      L = L < max_seq ? L : max_seq;
      const PrefillRange r = prefill_range(qlen, L, pg.by_U, ug);
      if (4 * ug < r.units) c[k] = r.n_steps > 0 ? r.n_steps : 1;
    }
    sum += c[k];
    if constexpr (STATS) {
      mx = c[k] > mx ? c[k] : mx;
      n += __popcll(__ballot(c[k] > 0));  // of the wave
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if constexpr (STATS) mx = wave_reduce(mx, [](int a, int b) { return a > b ? a : b; });
  if (lane == 63) {
    red[wave] = incl;
    if constexpr (STATS) {
      red[kPrefillWaves + wave] = mx;
      red[2 * kPrefillWaves + wave] = n;
    }
  }
  __syncthreads();
  int base = incl - sum;
  PrefillLine line{0, 0, 0};
#pragma unroll
  for (int w = 0; w < kPrefillWaves; ++w) {
    if (w < wave) base += red[w];
    line.total += red[w];
    if constexpr (STATS) {
      line.longest = red[kPrefillWaves + w] > line.longest ? red[kPrefillWaves + w] : line.longest;
      line.groups += red[2 * kPrefillWaves + w];
    }
  }
#pragma unroll
  for (int k = 0; k < kPrefillEntries / (64 * kPrefillWaves); ++k)
    if (k < per && e0 + k < E) {
      pfx[e0 + k] = base;
      base += c[k];
    }
  if (threadIdx.x == 0) pfx[E] = line.total;
  __syncthreads();
  return PrefillLine{__builtin_amdgcn_readfirstlane(line.total), __builtin_amdgcn_readfirstlane(line.longest),
                     __builtin_amdgcn_readfirstlane(line.groups)};
}

// First step of workgroup w's share of T steps over W workgroups (the callers
// take W <= T, so that every share has a step: a part's slot is then written
// by its workgroup whenever the merge reads it).
__device__ __forceinline__ int64_t prefill_share(int w, int64_t T, int W) { return w * T / W; }

// A part's partial of one unit: D/32 x 4 runs of 64 lanes x 4 fp32 (the
// output accumulators as the lanes hold them, so both the store and the
// merge's load are whole 1 KB wave accesses), then the 32 queries' reference
// maxima (log2 domain) and sums. Workgroup w owns partial slots 2 w (its first
// unit group) and 2 w + 1 (a later one), four units each. Behind the slots of
// the grid's W workgroups: the number that did share (an int), for the merge.
template <int D>
constexpr int prefill_part_floats() {
  return 32 * D + 64;
}
constexpr int kShareTailBytes = 16;
template <int D>
__device__ __forceinline__ int *prefill_shared_by(float *part, int W) {
  return reinterpret_cast<int *>(part + static_cast<int64_t>(W) * 2 * 4 * prefill_part_floats<D>());
}

// The attention kernel's arguments: one struct, the kernel's only parameter
// (prefill_args reads it from the kernel-argument segment).
struct PrefillArgs {
  const uint8_t *kc, *vc;
  const float *ksc, *vsc;
  const uint16_t *q;
  int64_t q_st, q_sh;
  uint16_t *out;
  int64_t o_st, o_sh;
  const int32_t *cu_q, *seq_lens, *bt;
  int64_t bt_stride;
  int Mb, max_seq, Hkv, BS, nb;
  float scale_log2;
  FastDiv by_BS;
  PrefillGrid pg;
  float *part;
  const float *sinks;
};

// The kernel's arguments, read again from the kernel-argument segment (the
// pointer is opaque to the compiler). A shared launch's loop over unit groups
// calls this per group: with the arguments live across the loop instead, some
// 70 scalar registers spill into the key loop (a 64-key step then takes 1.39
// us against 0.99).
__device__ __forceinline__ const PrefillArgs &prefill_args() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const PrefillArgs *)(p);
}

// A float at an address that every lane shares, by a scalar load: the compiler
// takes the pointers of the argument struct as writable in the key loop, and a
// vector load there counts with the copies in flight and waits for them (a
// 512-token fp8 prompt at 32/8 heads 23.2 us so, 21.8 with scalar loads).
__device__ __forceinline__ float load_scalar(const float *p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) float *>(reinterpret_cast<uintptr_t>(p));
}

// SHARED: workgroups share the launch's steps evenly (PrefillGrid::W), else one per unit group.
// SPAN: unit groups may span query tiles (PrefillGrid::by_U).
template <int D, bool FP8, bool SHARED, bool SPAN>
__global__ __launch_bounds__(64 * kPrefillWaves, 2) void prefill_gqa_kernel(PrefillArgs kernel_args) {
  using LT = LdsTile<D>;
  static_assert(kPrefillWaves == 4, "one tile per wave per 64-key step");
  static_assert(D % 64 == 0, "whole copies per lane");
  constexpr int KB = LT::KB, VB = LT::VB;   // bytes of one bf16 tile's K, V
  constexpr int ESZ = FP8 ? 1 : 2;          // cache bytes per element
  constexpr int NC = D * 16 * ESZ / 1024;   // 16-byte copies per lane of a tile's K (and of its V)
  constexpr int DV = D / 64;                // bf16 V copies per token octet
  constexpr int SB = FP8 ? D * 16 : 16;     // fp8 staging bytes per tile, K or V
  __shared__ __attribute__((aligned(16))) uint8_t ldsk[2 * 4 * KB];  // bf16 K: two step slots of four tiles
  __shared__ __attribute__((aligned(16))) uint8_t ldsv[2 * 4 * VB];  // bf16 V: two step slots
  __shared__ __attribute__((aligned(16))) uint8_t stgk[4 * SB];      // fp8 K as copied, a tile per wave
  __shared__ __attribute__((aligned(16))) uint8_t stgv[4 * SB];      // fp8 V as copied
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, n = lane & 31, hh = lane >> 5;
  int id = blockIdx.x;
  // One argument of every 64-byte line, together: the lines come from memory in
  // one round trip, and the later argument reads hit the scalar cache (taken as
  // they are needed, the lines' misses stand one after another before the
  // first load of the queries).
  // (not volatile: that would count as a write, and loads after it as vector loads)
  asm("" : "+s"(id) : "s"(kernel_args.kc), "s"(kernel_args.o_sh), "s"(kernel_args.pg.n_ug), "s"(kernel_args.sinks));
  int b, kvh, ug, s_begin = 0;
  int part_slot = 0;       // SHARED: this workgroup's partial slot of the unit group (odd past its first)
  int64_t steps_left = 0;  // SHARED: of this workgroup's share
  if constexpr (SHARED) {
    const PrefillArgs &a = prefill_args();
    const PrefillGrid pg = a.pg;
    int *pfx = reinterpret_cast<int *>(ldsk);
    static_assert((kPrefillEntries + 1 + 3 * kPrefillWaves) * 4 <= 2 * 4 * KB, "the prefix fits the K slots");
    const int E = pg.batch * pg.n_ug;
    const PrefillLine line = prefill_prefix<true>(pfx, pfx + kPrefillEntries + 1, a.cu_q, a.seq_lens, a.max_seq, pg);
    const int total = line.total;
    const int64_t T = static_cast<int64_t>(total) * a.Hkv;
    int W = pg.W;
    if (!pg.forced)
      W = share_workgroups<D, FP8, true>(static_cast<float>(T), static_cast<float>(line.longest),
                                         static_cast<float>(line.groups) * static_cast<float>(a.Hkv), pg.W);
    W = __builtin_amdgcn_readfirstlane(W);
    if (id == 0 && threadIdx.x == 0) *prefill_shared_by<D>(a.part, pg.W) = W;
    int e;
    if (W > 0) {
      // XCD i mod 8 takes a contiguous eighth of the line: its workgroups read the same keys.
      if (id >= W) return;
      const int w = (id & 7) * (W / 8) + id / 8;
      W = T < W ? static_cast<int>(T) : W;
      if (w >= W) return;
      const int64_t x0 = prefill_share(w, T, W);
      steps_left = prefill_share(w + 1, T, W) - x0;
      kvh = static_cast<int>(x0 / total);
      const int y = static_cast<int>(x0 - static_cast<int64_t>(kvh) * total);
      int lo = 0, hi = E;  // the last entry with pfx <= y (entries of no steps share their successor's prefix)
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pfx[mid] <= y) lo = mid; else hi = mid;
      }
      e = __builtin_amdgcn_readfirstlane(lo);
      s_begin = __builtin_amdgcn_readfirstlane(y - pfx[e]);
      part_slot = 2 * w;
    } else {
      // A whole unit group each, the latest query tiles first.
      const int n = E * a.Hkv, g = (id & 7) * ((n + 7) / 8) + id / 8;
      if (id / 8 >= (n + 7) / 8 || g >= n) return;
      kvh = g / E;
      e = E - 1 - (g - kvh * E);
      steps_left = __builtin_amdgcn_readfirstlane(pfx[e + 1] - pfx[e]);
      if (steps_left <= 0) return;
    }
    b = e / pg.by_ug;
    ug = e - b * pg.n_ug;
  } else {
    const PrefillGrid &pg = kernel_args.pg;
    // Eight sub-items (item, share r of its unit groups) run at a time, one per XCD.
    const int q = (id >> 3) / pg.by_inner, r = (id >> 3) - q * pg.by_inner.d;
    int oct = pg.mixed ? r : q;
    const int inner = pg.mixed ? q : r;
    if (pg.mixed && (pg.by_inner.d & 1) == 0) {  // an even number of them: each row of the turn begins one further
      oct = r + q - q / pg.by_inner * pg.by_inner.d;
      oct = oct >= pg.by_inner.d ? oct - pg.by_inner.d : oct;
    }
    const int sub = 8 * oct + (id & 7);
    if (sub >= pg.n_sub) return;
    const int item = sub >> pg.log2R;
    ug = pg.n_ug - 1 - ((inner << pg.log2R) + (sub & (pg.R - 1)));
    if (ug < 0) return;
    b = item / pg.by_Hkv;
    kvh = item - b * pg.by_Hkv.d;
  }
  for (;;) {  // SHARED: the unit groups of the share; else one
  const PrefillArgs *ap = &kernel_args;
  if constexpr (SHARED) ap = &prefill_args();
  const uint8_t *__restrict__ const kc = ap->kc, *__restrict__ const vc = ap->vc;
  const float *__restrict__ const ksc = ap->ksc, *__restrict__ const vsc = ap->vsc;
  const int32_t *__restrict__ const cu_q = ap->cu_q;
  const FastDiv U = ap->pg.by_U;
  const int G = ap->pg.G;
  const int Hkv = ap->Hkv, BS = ap->BS, Mb = ap->Mb, nb = ap->nb;
  const float scale_log2 = ap->scale_log2;
  b = __builtin_amdgcn_readfirstlane(b);
  kvh = __builtin_amdgcn_readfirstlane(kvh);
  ug = __builtin_amdgcn_readfirstlane(ug);
  const int q0 = cu_q[b], q1 = cu_q[b + 1];
  int L = ap->seq_lens[b];
  const int qlen = q1 - q0;
  L = L < ap->max_seq ? L : ap->max_seq;
  PrefillRange rg = prefill_range(qlen, L, U, ug);
  rg.units = __builtin_amdgcn_readfirstlane(rg.units);
  rg.kend = __builtin_amdgcn_readfirstlane(rg.kend);
  rg.n_steps = __builtin_amdgcn_readfirstlane(rg.n_steps);
  if (4 * ug < rg.units) {  // else no query: the whole workgroup goes on together
  const int all_steps = rg.n_steps > 0 ? rg.n_steps : 1;  // as the shared line counts them
  int take = all_steps - s_begin;
  if constexpr (SHARED) {
    take = steps_left < take ? static_cast<int>(steps_left) : take;
    __syncthreads();  // the LDS of the unit group before (or of the prefix) is free
  }
  const bool partial = SHARED && take < all_steps;
  const int unit = 4 * ug + wave < rg.units ? 4 * ug + wave : rg.units - 1;
  const int qt = __builtin_amdgcn_readfirstlane(unit / U);
  const int t0 = qt * 32;
  // an idle wave (past the units, or a unit without a head) still copies its tile of every step
  const bool active = 4 * ug + wave == unit && unit - qt * U.d < G;
  const int h = kvh * G + (active ? unit - qt * U.d : 0);
  const int ctx = L - qlen;
  // Q^T operand j: lane l holds d = 16 j + 8 (l/32) .. + 7 of query t0 + l % 32.
  bf16x8 qb[D / 16];
  {
    const int tok = t0 + n;
    const bool valid = active && tok < qlen;
    const uint16_t *qp =
        ap->q + static_cast<int64_t>(q0 + (tok < qlen ? tok : t0)) * ap->q_st + static_cast<int64_t>(h) * ap->q_sh;
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
      u32x4 w = *reinterpret_cast<const u32x4 *>(qp + 16 * j + 8 * hh);
      if (!valid) w = u32x4{0u, 0u, 0u, 0u};
      qb[j] = __builtin_bit_cast(bf16x8, w);
    }
  }
  floatx16 o[D / 32];
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[c][r] = 0.f;
  float m_ref = -INFINITY, l_part = 0.f;

  // The steps taken here; key and query positions from here on count from their first key.
  const int key0 = 64 * s_begin;
  const int kend = rg.kend - key0;
  const int n_steps = rg.n_steps - s_begin < take ? rg.n_steps - s_begin : take;
  const int n_tiles = (kend + 15) / 16 < 4 * n_steps ? (kend + 15) / 16 : 4 * n_steps;
  const int region = D * BS * ESZ;
  const int min_pos = ctx + t0 - key0;  // the smallest query position of the wave
  // One past the last key any query of this wave sees: below kend where the unit
  // group goes on to later query tiles, whose keys must not reach this wave's
  // products (a masked key's probability is 0, but 0 times a V that is not finite is NaN).
  const int wend = min_pos + 32 < kend ? min_pos + 32 : kend;

  // Copy k of lane l moves piece p = 64 k + l of the wave's tile's K or V
  // (LDS offset 16 p). K piece p (both dtypes: 16-byte chunks): chunk p >> 4,
  // token p & 15, at ((p >> 4) BS + (p & 15)) 16 of the (block, head) K region
  // = lane part ((l >> 4) BS + (l & 15)) 16 + copy part 64 BS k. bf16 V piece
  // p: row p % D, octet p / D, at (p % D) BS 2 + 16 (p / D) = lane part 2 BS l
  // + copy part 128 BS (k % DV) + 16 (k / DV). fp8 V piece p: row p, at p BS =
  // lane part BS l + copy part 64 BS k. The tile's first token o0 goes into
  // the base.
  const uint32_t lane_k = static_cast<uint32_t>(((lane >> 4) * BS + (lane & 15)) * 16);
  const uint32_t lane_v = static_cast<uint32_t>(lane * BS * ESZ);
  const uint32_t ldsk0 = lds_addr(ldsk), ldsv0 = lds_addr(ldsv);
  const uint32_t stgk0 = lds_addr(stgk), stgv0 = lds_addr(stgv);
  float ks_next = 1.f, vs_next = 1.f, vs_stage = 1.f;  // fp8 scales: last K issued, its V, the staged V
  const int32_t *btrow = ap->bt + b * ap->bt_stride;
  const FastDiv by_BS = ap->by_BS;
  int bix = (key0 + 16 * wave) / by_BS;
  int o0 = key0 + 16 * wave - bix * BS;
  const int dbix = 64 / by_BS, do0 = 64 - dbix * BS;
  int wbase = bix;  // the window: lane i holds the id of block wbase + i
  int win = load_i32_drained(btrow, wbase + lane, Mb);
  int64_t vbase = 0;  // V of the wave's tile of the step whose K went out last: cache offset
  auto has_tile = [&](int s) { return s < n_steps && 4 * s + wave < n_tiles; };  // uniform
  // K of the wave's tile of step s into K slot `slot` (fp8: into the staging area)
  auto issue_k = [&](int s, int slot) {
    if (has_tile(s)) {
      if (bix - wbase >= 64) {  // at most once per 64 blocks (its wait drains the copies in flight)
        wbase += 64;
        win = load_i32_drained(btrow, wbase + lane, Mb);
      }
      int blk = __builtin_amdgcn_readlane(win, bix - wbase);
      if (!(blk >= 0 && blk < nb)) blk = 0;
      const int64_t rb = static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(blk * Hkv + kvh)) *
                                              static_cast<uint32_t>(region));
      vbase = rb + o0 * ESZ;
      if constexpr (FP8) {
        ks_next = load_scalar(ksc + blk * Hkv + kvh);
        vs_next = load_scalar(vsc + blk * Hkv + kvh);
      }
      // copy part of K copy k: 64 BS k = 1024 k (its LDS offset, the instruction
      // offset) + k (64 BS - 1024)
      uint32_t kst = static_cast<uint32_t>(64 * BS);
      asm volatile("" : "+s"(kst));
      const __amdgpu_buffer_rsrc_t kr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(kc + rb + o0 * 16), 0, region, kRawBufferWord3);
      const uint32_t dst = FP8 ? stgk0 + static_cast<uint32_t>(wave * SB)
                               : ldsk0 + static_cast<uint32_t>((4 * slot + wave) * KB);
      buffer_copy16_run_to_lds<NC>(kr, lane_k, kst - 1024u, dst);
    }
    o0 += do0;
    bix += dbix;
    if (o0 >= BS) {
      o0 -= BS;
      ++bix;
    }
  };
  // V of the wave's tile of step s (whose K went out last) into V slot `slot`
  auto issue_v = [&](int s, int slot) {
    if (has_tile(s)) {
      const __amdgpu_buffer_rsrc_t vr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(vc + vbase), 0, region, kRawBufferWord3);
      if constexpr (FP8) {
        vs_stage = vs_next;
        const uint32_t dst = stgv0 + static_cast<uint32_t>(wave * SB);
        uint32_t vst = static_cast<uint32_t>(64 * BS);
        asm volatile("" : "+s"(vst));
#pragma unroll
        for (int k = 0; k < NC; ++k) buffer_copy16_to_lds(vr, lane_v, vst * k, dst + 1024 * k);
      } else {
        const uint32_t dst = ldsv0 + static_cast<uint32_t>((4 * slot + wave) * VB);
        uint32_t vst = static_cast<uint32_t>(128 * BS);
        asm volatile("" : "+s"(vst));
#pragma unroll
        for (int k = 0; k < NC; ++k)
          buffer_copy16_to_lds(vr, lane_v, vst * (k % DV) + 16 * (k / DV), dst + 1024 * k);
      }
    }
  };
  // fp8: the wave's K tile, staged, into bf16 K slot `slot` at scale sc.
  // Piece p = 64 i + l: chunk c = p >> 4 (16 d), token m = p & 15 -> bf16
  // chunks 2c, 2c + 1 of token m.
  auto convert_k = [&](float sc, int slot) {
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
      const int pc = 64 * i + lane;
      const u32x4 w = *reinterpret_cast<const u32x4 *>(stgk + wave * SB + pc * 16);
      uint8_t *dk = ldsk + (4 * slot + wave) * KB + ((2 * (pc >> 4)) * 16 + (pc & 15)) * 16;
      *reinterpret_cast<u32x4 *>(dk) = fp8x8_to_bf16_words(w[0], w[1], sc);
      *reinterpret_cast<u32x4 *>(dk + 256) = fp8x8_to_bf16_words(w[2], w[3], sc);
    }
  };
  // fp8: the wave's V tile, staged, into bf16 V slot `slot` at scale sc,
  // tokens at or past vt zeroed (the slots past the keys may hold NaN). Piece
  // p = 64 i + l: row p, 16 tokens -> octets 0, 1 of row p.
  auto convert_v = [&](float sc, int vt, int slot) {
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
      const int pc = 64 * i + lane;
      const u32x4 w = *reinterpret_cast<const u32x4 *>(stgv + wave * SB + pc * 16);
      u32x4 lo = fp8x8_to_bf16_words(w[0], w[1], sc), hi = fp8x8_to_bf16_words(w[2], w[3], sc);
      if (vt < 16) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (e >= vt) lo[e >> 1] &= (e & 1) ? 0x0000FFFFu : 0xFFFF0000u;
          if (8 + e >= vt) hi[e >> 1] &= (e & 1) ? 0x0000FFFFu : 0xFFFF0000u;
        }
      }
      uint8_t *dv = ldsv + (4 * slot + wave) * VB;
      *reinterpret_cast<u32x4 *>(dv + pc * 16) = lo;
      *reinterpret_cast<u32x4 *>(dv + (D + pc) * 16) = hi;
    }
  };
  // Step s's copies have landed (this wave's): make its V tile (and fp8: the
  // next step's K tile) ready in the bf16 slots -- fp8 conversion, slots of a
  // partial tile past the keys zeroed.
  // Before the last step every wave's tile of step s is whole and its K tile
  // of step s + 1 is converted whether or not it exists (a tile past the keys
  // is masked): the fp8 conversion then runs without branches, its four LDS
  // reads ahead of the conversions.
  auto land_body = [&](int s) {
    if constexpr (FP8) {
      u32x4 wv[D / 64], wk[D / 64];
#pragma unroll
      for (int i = 0; i < D / 64; ++i) {
        wv[i] = *reinterpret_cast<const u32x4 *>(stgv + wave * SB + (64 * i + lane) * 16);
        wk[i] = *reinterpret_cast<const u32x4 *>(stgk + wave * SB + (64 * i + lane) * 16);
      }
      uint8_t *dv = ldsv + (4 * (s & 1) + wave) * VB;
      uint8_t *dk = ldsk + (4 * ((s + 1) & 1) + wave) * KB;
#pragma unroll
      for (int i = 0; i < D / 64; ++i) {
        const int pc = 64 * i + lane;
        *reinterpret_cast<u32x4 *>(dv + pc * 16) = fp8x8_to_bf16_words(wv[i][0], wv[i][1], vs_stage);
        *reinterpret_cast<u32x4 *>(dv + (D + pc) * 16) = fp8x8_to_bf16_words(wv[i][2], wv[i][3], vs_stage);
        uint8_t *k = dk + ((2 * (pc >> 4)) * 16 + (pc & 15)) * 16;
        *reinterpret_cast<u32x4 *>(k) = fp8x8_to_bf16_words(wk[i][0], wk[i][1], ks_next);
        *reinterpret_cast<u32x4 *>(k + 256) = fp8x8_to_bf16_words(wk[i][2], wk[i][3], ks_next);
      }
    }
  };
  auto land = [&](int s) {
    int vt = kend - 64 * s - 16 * wave;  // keys of this wave's tile of step s
    vt = vt < 0 ? 0 : (vt > 16 ? 16 : vt);
    if constexpr (FP8) {
      if (vt > 0) convert_v(vs_stage, vt, s & 1);  // uniform
      if (has_tile(s + 1)) convert_k(ks_next, (s + 1) & 1);
    } else if (vt > 0 && vt < 16) {  // uniform; at most once per workgroup
#pragma unroll
      for (int i = 0; i < D / 32; ++i) {
        const int pc = 64 * i + lane;
        const int cnt = vt - 8 * (pc / D);
        u32x4 *ptr = reinterpret_cast<u32x4 *>(ldsv + (4 * (s & 1) + wave) * VB + pc * 16);
        u32x4 w = *ptr;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e >= cnt) w[e >> 1] &= (e & 1) ? 0x0000FFFFu : 0xFFFF0000u;
        *ptr = w;
      }
    }
  };
  const int kn = (n & 16) | (((n >> 2) & 3) == 1 ? (n & 3) + 8 : ((n >> 2) & 3) == 2 ? (n & 3) + 4 : (n & 15));
  const bf16x2 ones = __builtin_bit_cast(bf16x2, 0x3F803F80u);
  uint32_t pw[4][4];  // PV B operands of the step being finished: packed bf16 probabilities

  // S^T of step s (K slot s & 1) into (x0, x1)
  auto qk = [&](int s, floatx16 &x0, floatx16 &x1) {
#pragma unroll
    for (int r = 0; r < 16; ++r) x0[r] = x1[r] = 0.f;
    const uint8_t *lk = ldsk + ((s & 1) * 4 + (kn >> 4)) * KB + (kn & 15) * 16;
#pragma unroll
    for (int jj = 0; jj < D / 16; ++jj) {
      const bf16x8 a0 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(lk + (2 * jj + hh) * 256));
      const bf16x8 a1 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(lk + 2 * KB + (2 * jj + hh) * 256));
      x0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, qb[jj], x0, 0, 0, 0);
      x1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, qb[jj], x1, 0, 0, 0);
    }
  };
  // causal / end mask of step s's scores
  auto mask = [&](int s, floatx16 &x0, floatx16 &x1) {
    const int kb = 64 * s;
    if (!(kend >= kb + 64 && kb + 63 <= min_pos)) {  // uniform: masks in this step
      const int pos = min_pos + n;
      const int lim = (pos < kend - 1 ? pos : kend - 1) - kb - 8 * hh;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (16 * (r / 8) + (r % 8) > lim) x0[r] = -INFINITY;
        if (32 + 16 * (r / 8) + (r % 8) > lim) x1[r] = -INFINITY;
      }
    }
  };
  // exponents against the reference maximum and their maximum
  auto expo = [&](floatx16 &x0, floatx16 &x1) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      x0[r] = __builtin_fmaf(x0[r], scale_log2, -m_ref);
      x1[r] = __builtin_fmaf(x1[r], scale_log2, -m_ref);
    }
    float mt0 = fmaxf(x0[0], x0[1]), mt1 = fmaxf(x1[0], x1[1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) {
      mt0 = fmaxf(fmaxf(mt0, x0[r]), x0[r + 1]);
      mt1 = fmaxf(fmaxf(mt1, x1[r]), x1[r + 1]);
    }
    float mt = fmaxf(mt0, mt1);
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
    return fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
  };
  // the rare move of the reference maximum (after the PV products of the steps before)
  auto rescale = [&](float mt, floatx16 &x0, floatx16 &x1) {
    const bool move = mt > SOFTMAX_TAU;
    if (__any(move)) {
      const float sh = move ? mt : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        x0[r] -= sh;
        x1[r] -= sh;
      }
      const float corr = fast_exp2(-sh);
      l_part *= corr;
      m_ref += sh;
#pragma unroll
      for (int c = 0; c < D / 32; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[c][r] *= corr;
    }
  };
  // probabilities, packed as the PV operands, and their row sum
  auto probs = [&](floatx16 &x0, floatx16 &x1) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      x0[r] = fast_exp2(x0[r]);
      x1[r] = fast_exp2(x1[r]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const floatx16 &sv = t < 2 ? x0 : x1;
      const int e0 = 8 * (t & 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) pw[t][i] = pack_bf16x2(sv[e0 + 2 * i], sv[e0 + 2 * i + 1]);
    }
    float ps = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        ps = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pw[t][i]), ones, ps, false);
    l_part += ps;
  };
  // P V^T of step s (V slot s & 1); tiles past the keys skipped when `partial`
  auto pv = [&](int s, bool partial) {
    const uint8_t *lv = ldsv + (s & 1) * 4 * VB + hh * D * 16 + n * 16;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (partial && kend - 64 * s - 16 * t <= 0) continue;  // uniform
      const bf16x8 pb = __builtin_bit_cast(bf16x8, (u32x4{pw[t][0], pw[t][1], pw[t][2], pw[t][3]}));
#pragma unroll
      for (int c = 0; c < D / 32; ++c) {
        const u32x4 w = *reinterpret_cast<const u32x4 *>(lv + t * VB + 32 * c * 16);
        o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), pb, o[c], 0, 0, 0);
      }
    }
  };
  // The same with the keys at or past the wave's last left out: tiles skipped,
  // the slots of its partial tile zeroed in the operand.
  auto pv_end = [&](int s) {
    const uint8_t *lv = ldsv + (s & 1) * 4 * VB + hh * D * 16 + n * 16;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int left = wend - 64 * s - 16 * t;  // keys of the tile that the wave sees
      if (left <= 0) continue;                  // uniform
      const bf16x8 pb = __builtin_bit_cast(bf16x8, (u32x4{pw[t][0], pw[t][1], pw[t][2], pw[t][3]}));
      u32x4 seen;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        seen[i] = (8 * hh + 2 * i < left ? 0xFFFFu : 0u) | (8 * hh + 2 * i + 1 < left ? 0xFFFF0000u : 0u);
#pragma unroll
      for (int c = 0; c < D / 32; ++c) {
        const u32x4 w = *reinterpret_cast<const u32x4 *>(lv + t * VB + 32 * c * 16) & seen;
        o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), pb, o[c], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // One step of the pipeline: finish step s (its scores in c0, c1 are
  // exponents against the reference) while scoring step s + 1 into n0, n1.
  auto body = [&](int s, floatx16 &c0, floatx16 &c1, floatx16 &n0, floatx16 &n1) {
    wait_vmcnt<0>();  // this wave's copies of step s's V and step s + 1's K
    land_body(s);
    barrier_lds();    // ... every wave's; every wave is done with step s - 1
    issue_v(s + 1, (s + 1) & 1);
    issue_k(s + 2, s & 1);
    {  // an idle wave computes on zero queries and stores nothing
      qk(s + 1, n0, n1);
      probs(c0, c1);
      // keeps the probabilities in this block (ahead of the mask's branch)
      asm volatile("" ::"v"(l_part), "v"(pw[0][0]), "v"(pw[0][1]), "v"(pw[0][2]), "v"(pw[0][3]), "v"(pw[1][0]),
                   "v"(pw[1][1]), "v"(pw[1][2]), "v"(pw[1][3]), "v"(pw[2][0]), "v"(pw[2][1]), "v"(pw[2][2]),
                   "v"(pw[2][3]), "v"(pw[3][0]), "v"(pw[3][1]), "v"(pw[3][2]), "v"(pw[3][3]));
      // the score products of step s + 1 interleaved with step s's probabilities
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // LDS reads, four ahead
#pragma unroll
      for (int i = 0; i < 2 * D / 16; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        if (i + 4 < 2 * D / 16) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // VALU
      }
      mask(s + 1, n0, n1);
      const float mt = expo(n0, n1);
      pv(s, false);
      // step s's PV products interleaved with step s + 1's exponents
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // LDS reads, four ahead
#pragma unroll
      for (int i = 0; i < 4 * D / 32; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        if (i + 4 < 4 * D / 32) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
      }
      rescale(mt, n0, n1);
    }
  };

  if (n_steps > 0) {
    issue_k(0, 0);
    if constexpr (FP8) {
      wait_vmcnt<0>();
      if (has_tile(0)) convert_k(ks_next, 0);
    }
    issue_v(0, 0);
    issue_k(1, 1);
    if constexpr (!FP8) {
      if (has_tile(1)) wait_vmcnt<2 * NC>(); else wait_vmcnt<NC>();  // K of step 0 landed
    }
    barrier_lds();
    floatx16 a0, a1, b0, b1;
    {
      qk(0, a0, a1);
      mask(0, a0, a1);
      // the reference maximum starts at the first step's row maximum (a query
      // that sees no key of it -- only past the unit group's first -- sees none at all)
      float mt = fmaxf(a0[0], a1[0]);
#pragma unroll
      for (int r = 1; r < 16; ++r) mt = fmaxf(mt, fmaxf(a0[r], a1[r]));
      const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
      mt = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1])) * scale_log2;
      m_ref = mt == -INFINITY ? 0.f : mt;
      rescale(expo(a0, a1), a0, a1);
    }
    // the last step: its V, its probabilities, its PV products (tiles past the keys skipped)
    auto tail = [&](int s, floatx16 &c0, floatx16 &c1) {
      wait_vmcnt<0>();
      land(s);
      barrier_lds();
      probs(c0, c1);
      pv(s, true);
    };
    const int n_body = n_steps - 1;
    int s = 0;
    if constexpr (!SPAN) {
      for (; s + 2 <= n_body; s += 2) {
        body(s, a0, a1, b0, b1);
        body(s + 1, b0, b1, a0, a1);
      }
      if (s < n_body) {
        body(s, a0, a1, b0, b1);
        tail(s + 1, b0, b1);
      } else {
        tail(s, a0, a1);
      }
    } else {
      // A wave whose keys end before the steps do stops its products with the
      // step that holds its last key; its copies go on as the others'.
      const bool ends = wend < kend && wend < 64 * n_steps;  // uniform
      const int n_whole = ends && wend < 64 * n_body ? (wend > 0 ? wend >> 6 : 0) : n_body;
      for (; s + 2 <= n_whole; s += 2) {
        body(s, a0, a1, b0, b1);
        body(s + 1, b0, b1, a0, a1);
      }
      if (s < n_whole) {
        body(s, a0, a1, b0, b1);
        ++s;
        a0 = b0;
        a1 = b1;
      }
      if (!ends) {
        tail(s, a0, a1);
      } else {
        const int s_last = s;
        for (; s < n_steps; ++s) {
          wait_vmcnt<0>();
          if (s < n_body) {
            land_body(s);
            barrier_lds();
            issue_v(s + 1, (s + 1) & 1);
            issue_k(s + 2, s & 1);
          } else {
            land(s);
            barrier_lds();
          }
          if (s == s_last) {
            probs(a0, a1);
            pv_end(s);
          }
        }
      }
    }
  }
  if (active) {
  const PrefillArgs *ae = &kernel_args;  // SHARED: the epilogue's arguments are not held through the key loop
  if constexpr (SHARED) ae = &prefill_args();
  float l = l_part;
  {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  if (partial) {  // uniform
    float *pp = ae->part + (static_cast<int64_t>(part_slot) * 4 + wave) * prefill_part_floats<D>();
#pragma unroll
    for (int c = 0; c < D / 32; ++c)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<floatx4 *>(pp + ((4 * c + g) * 64 + lane) * 4) =
            floatx4{o[c][4 * g], o[c][4 * g + 1], o[c][4 * g + 2], o[c][4 * g + 3]};
    // a query that saw no key of this part must not set the merged maximum
    if (hh == 0) {
      pp[32 * D + n] = l > 0.f ? m_ref : -INFINITY;
      pp[32 * D + 32 + n] = l;
    }
  } else if (t0 + n < qlen) {
    // An attention sink (a zero-value logit of head h, natural-log units) adds
    // its weight against the row's reference maximum to the denominator.
    if (ae->sinks != nullptr) l += exp2f(ae->sinks[h] * 1.4426950408889634f - m_ref);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t *const op = ae->out + static_cast<int64_t>(q0 + t0 + n) * ae->o_st + static_cast<int64_t>(h) * ae->o_sh;
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {  // d = 32 c + 8 g + 4 hh + 0..3
        const u32x2 w = {pack_bf16x2(o[c][4 * g] * inv, o[c][4 * g + 1] * inv),
                         pack_bf16x2(o[c][4 * g + 2] * inv, o[c][4 * g + 3] * inv)};
        *reinterpret_cast<u32x2 *>(op + 32 * c + 8 * g + 4 * hh) = w;
      }
    }
  }
  }
  if constexpr (SHARED) {
    steps_left -= take;
    part_slot |= 1;
  }
  }
  if constexpr (!SHARED) break;
  if (steps_left <= 0) break;
  s_begin = 0;
  const PrefillArgs &an = prefill_args();
  if (++ug == an.pg.n_ug) {
    ug = 0;
    if (++b == an.pg.batch) {
      b = 0;
      if (++kvh == an.Hkv) break;  // never with steps left
    }
  }
  }
}

// Log-sum-exp merge of a shared launch's partials: one wave per unit and 32
// output columns (blockIdx.y), in the lanes' accumulator layout of the
// attention kernel; a unit group that one workgroup took whole was finished
// there. Bound by reading the partials (66 KB per part at d=128).
template <int D>
__global__ __launch_bounds__(64 * kPrefillWaves) void prefill_merge_kernel(
    float *__restrict__ part, uint16_t *__restrict__ out, int64_t o_st, int64_t o_sh,
    const int32_t *__restrict__ cu_q, const int32_t *__restrict__ seq_lens, int max_seq, int Hkv, PrefillGrid pg,
    const float *__restrict__ sinks) {
  constexpr int PF = prefill_part_floats<D>();
  __shared__ int pfx[kPrefillEntries + 1];
  __shared__ int red[kPrefillWaves];
  const int by = *prefill_shared_by<D>(part, pg.W);  // (on its way while the prefix is formed)
  const int total = prefill_prefix<false>(pfx, red, cu_q, seq_lens, max_seq, pg).total;
  const int shared_by = __builtin_amdgcn_readfirstlane(by);
  if (shared_by == 0) return;  // every unit group was taken whole
  const int E = pg.batch * pg.n_ug;
  const int kvh = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x / E));
  const int e = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x - kvh * E));
  const int c = blockIdx.y;
  const int b = __builtin_amdgcn_readfirstlane(e / pg.by_ug);
  const int ug = e - b * pg.n_ug;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, n = lane & 31, hh = lane >> 5;
  const int q0 = cu_q[b];
  const int qlen = cu_q[b + 1] - q0;
  const FastDiv U = pg.by_U;
  const int units = qlen > 0 ? ((qlen + 31) >> 5) * U.d : 0;
  const int unit = 4 * ug + wave;
  const int n_e = __builtin_amdgcn_readfirstlane(pfx[e + 1] - pfx[e]);
  if (n_e <= 0 || unit >= units) return;
  // The workgroups whose shares [share(w), share(w + 1)) meet this group's steps [x0, x0 + n_e).
  const int64_t T = static_cast<int64_t>(total) * Hkv;
  const int W = T < shared_by ? static_cast<int>(T) : shared_by;
  const int64_t x0 = static_cast<int64_t>(kvh) * total + __builtin_amdgcn_readfirstlane(pfx[e]);
  const int64_t x1 = x0 + n_e;
  int w0 = static_cast<int>(x0 * W / T);
  while (prefill_share(w0 + 1, T, W) <= x0) ++w0;
  while (prefill_share(w0, T, W) > x0) --w0;
  int w1 = w0;  // last
  while (prefill_share(w1 + 1, T, W) < x1) ++w1;
  w0 = __builtin_amdgcn_readfirstlane(w0);
  w1 = __builtin_amdgcn_readfirstlane(w1);
  if (w0 == w1) return;
  // The group is its workgroup's first unit group iff the share starts inside it (or with it).
  const float *p0 = part + ((2 * static_cast<int64_t>(w0) + (prefill_share(w0, T, W) < x0 ? 1 : 0)) * 4 + wave) * PF;
  const float *pn = part + (2 * static_cast<int64_t>(w0 + 1) * 4 + wave) * PF;  // the later parts, 8 PF apart
  const int np = w1 - w0;
  const int qt = __builtin_amdgcn_readfirstlane(unit / U);
  if (unit - qt * U.d >= pg.G) return;  // a unit without a head
  const int h = kvh * pg.G + (unit - qt * U.d);
  float M = p0[32 * D + n];
#pragma unroll 4
  for (int s = 0; s < np; ++s) M = fmaxf(M, pn[s * (8 * PF) + 32 * D + n]);
  const float m_use = M == -INFINITY ? 0.f : M;
  float l = 0.f;
  floatx4 acc[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) acc[g] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto add = [&](const float *ps) {
    const float w = exp2f(ps[32 * D + n] - m_use);
    l += w * ps[32 * D + 32 + n];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const floatx4 x = *reinterpret_cast<const floatx4 *>(ps + ((4 * c + g) * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[g][i] += w * x[i];
    }
  };
  add(p0);
#pragma unroll 4
  for (int s = 0; s < np; ++s) add(pn + s * (8 * PF));
  const int tok = 32 * qt + n;
  if (tok >= qlen) return;
  if (sinks != nullptr) l += exp2f(sinks[h] * 1.4426950408889634f - m_use);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t *op = out + static_cast<int64_t>(q0 + tok) * o_st + static_cast<int64_t>(h) * o_sh;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const u32x2 w = {pack_bf16x2(acc[g][0] * inv, acc[g][1] * inv), pack_bf16x2(acc[g][2] * inv, acc[g][3] * inv)};
    *reinterpret_cast<u32x2 *>(op + 32 * c + 8 * g + 4 * hh) = w;
  }
}

// The launch's grid. With a workspace (may_share), the steps may be shared over
// up to W workgroups where that is expected to be faster; share > 0 sets W.
static PrefillGrid prefill_grid(int batch, int Hkv, int G, int D, bool fp8, int max_query_len, int max_seq,
                                int share, bool may_share) {
  PrefillGrid pg;
  const int64_t n_qt = (static_cast<int64_t>(max_query_len) + 31) / 32;
  int U = G;
  pg.n_ug = static_cast<int>((n_qt * U + 3) / 4);
  pg.batch = batch;
  const int64_t items = static_cast<int64_t>(batch) * Hkv;
  const int64_t wgs = items * pg.n_ug;
  pg.W = 0;
  pg.forced = share > 0;
  if (may_share && static_cast<int64_t>(batch) * pg.n_ug <= kPrefillEntries) {
    if (share > 0) {
      pg.W = (share + 7) / 8 * 8;
    } else if (wgs < 4 * kPrefillCus && max_seq > kShareMinKeys) {
      const float steps = static_cast<float>(max_seq) / 64.f;
      const float qsteps = max_query_len < max_seq ? static_cast<float>(max_query_len) / 64.f : steps;
      // the host knows the longest lengths only: several sequences are taken
      // to bring 0.6 of the longest one's work on average
      const float T = static_cast<float>(wgs) * (steps - 0.5f * qsteps) * (batch > 1 ? 0.6f : 1.f);
      const auto choose = D == 128 ? (fp8 ? share_workgroups<128, true, false> : share_workgroups<128, false, false>)
                                   : (fp8 ? share_workgroups<64, true, false> : share_workgroups<64, false, false>);
      pg.W = choose(T, steps, static_cast<float>(wgs), 2 * kPrefillCus);
    }
  }
  // At most one unit group per CU with a tile's units to themselves (made up to
  // a multiple of four by units without a head), or two where three waves in
  // four or more then have a head: so, as the chip has room for them and no
  // group then runs on to a later tile's keys nor its waves on keys that they do
  // not see. Past that, packed: the idle waves cost more.
  // (us, packed -> not: one prompt of 512 at 16/8 heads bf16 20.9 -> 19.7, fp8
  // 23.0 -> 21.1; at 28/4 21.3 -> 20.6; 256 groups so, two prompts of 512 at 16/8
  // 22.2 -> 21.0; but 512 groups, four prompts, 25.2 -> 28.5. Over 26 to 38
  // shapes of 257 to 512 groups so, the time not packed against packed: 14/2
  // heads d=64 bf16 0.974, fp8 0.942; 28/4 bf16 0.984, fp8 0.996; but 16/8 1.018
  // and 0.993.)
  const int64_t tile_ug = (G + 3) / 4;
  const int per_cu = G >= 3 * tile_ug ? 2 : 1;
  if (pg.W == 0 && items * n_qt * tile_ug <= per_cu * kPrefillCus) {
    U = static_cast<int>(4 * tile_ug);
    pg.n_ug = static_cast<int>(n_qt * tile_ug);
  }
  // Items are dealt to the eight XCDs in turn: R makes the KV heads of one
  // sequence (its unit groups dealt over R XCDs where there are fewer than
  // eight) cover all of them, so that sequences of different lengths load the
  // XCDs alike (8 prompts of 438-1,314 tokens at 28/4 heads: 98 us so, 107
  // with two sequences at a time on four XCDs each).
  pg.R = 1;
  while (static_cast<int64_t>(Hkv) * pg.R % 8 != 0) pg.R *= 2;
  while (pg.R > 1 && pg.R > pg.n_ug) pg.R /= 2;
  pg.n_inner = (pg.n_ug + pg.R - 1) / pg.R;
  pg.n_sub = static_cast<int>(items * pg.R);
  pg.log2R = 0;
  while ((1 << pg.log2R) < pg.R) ++pg.log2R;
  pg.G = G;
  pg.by_U = fast_div(U);
  pg.by_ug = fast_div(pg.n_ug);
  // Up to three workgroups per CU, an XCD takes its sub-items in turn, the
  // longest chains of all of them first; past that one sub-item after another,
  // as their keys no longer stay in its L2 together. (us, after another -> in
  // turn: two prompts of 2,048 at 14/2 heads 42.4 -> 38.0, four of 1,500 48.8 ->
  // 41.1, two of 1,000 at 32/8 42.7 -> 39.2; but 1,024 workgroups, 16 of 256,
  // 38.8 -> 53.4.) The dispatcher deals an XCD's workgroups to its 32 CUs in turn
  // as well: an even number of sub-items would put each on the same few CUs
  // every time, the longest's among them, so the rows of the turn are rotated
  // (8 ragged prompts of 133-400 at 28/4 heads 23.9 -> 20.7, fp8 26.6 -> 22.4).
  // Over 192 shapes of 9 to 240 items of 50 to 2,000 tokens the turn takes 0.947 of
  // the time of one sub-item after another, 0.72 at best and 1.1 at worst (few ragged
  // sequences whose last round of workgroups ends up uneven).
  const int n_oct = (pg.n_sub + 7) / 8;
  // Prompts only: over cached contexts (more than an eighth) a chain's length
  // follows its sequence, the turn leaves the longest's tiles for last and the
  // XCD's keys outgrow its L2 (4 x 600 over 1,000-3,000 at 32/8 fp8 107.7 -> 134.6).
  const bool prompts = static_cast<int64_t>(8) * max_query_len >= static_cast<int64_t>(7) * max_seq;
  pg.mixed = prompts && n_oct > 1 && static_cast<int64_t>(8) * n_oct * pg.n_inner <= 3 * kPrefillCus;
  pg.by_inner = fast_div(pg.mixed ? n_oct : pg.n_inner);
  pg.by_Hkv = fast_div(Hkv);
  return pg;
}

static int64_t prefill_workspace(const PrefillGrid &pg, int D) {
  return pg.W > 0 ? static_cast<int64_t>(pg.W) * 2 * 4 * (32 * D + 64) * 4 + kShareTailBytes : 0;
}

}  // namespace wkv

using namespace wkv;

static int launch_prefill(const wkv_cache_t *cache, const void *key, int64_t key_stride_t, int64_t key_stride_h,
                          const void *value, int64_t value_stride_t, int64_t value_stride_h,
                          const int64_t *slot_mapping, int64_t num_tokens, const void *q, int64_t q_stride_t,
                          int64_t q_stride_h, void *out, int64_t out_stride_t, int64_t out_stride_h,
                          int32_t num_q_heads, const int32_t *cu_seqlens_q, const int32_t *seq_lens,
                          const int32_t *block_table, int64_t bt_stride, int32_t max_blocks_per_seq, int32_t batch,
                          int32_t max_query_len, int32_t max_seq_len, float scale, int32_t workgroups,
                          void *workspace, int64_t workspace_bytes, const float *sinks, void *stream) {
  int rc = check_cache(cache, -1);
  if (rc) return rc;
  WKV_CHECK_ARG(batch >= 0 && batch <= 65535, "batch must be in [0, 65535] (got %d)", batch);
  WKV_CHECK_ARG(num_tokens >= 0, "num_tokens must be >= 0");
  // The step's new tokens go into the cache first (same stream: the attention
  // launch below reads them back), once nothing is left to refuse.
  auto append = [&]() -> int {
    if (key == nullptr && value == nullptr && slot_mapping == nullptr) return WKV_OK;
    return cache->kv_dtype == WKV_KV_FP8_E4M3
               ? wkv_append_fp8(cache, key, key_stride_t, key_stride_h, value, value_stride_t, value_stride_h,
                                slot_mapping, num_tokens, stream)
               : wkv_append(cache, key, key_stride_t, key_stride_h, value, value_stride_t, value_stride_h,
                            slot_mapping, num_tokens, stream);
  };
  if (batch == 0 || max_query_len == 0) return append();
  const int Hkv = cache->num_kv_heads, D = cache->head_dim, BS = cache->block_size;
  WKV_CHECK_ARG(num_q_heads > 0 && num_q_heads % Hkv == 0, "num_q_heads %d must be a multiple of num_kv_heads %d",
                num_q_heads, Hkv);
  const int G = num_q_heads / Hkv;
  WKV_CHECK_ARG(cache->num_blocks * Hkv <= INT32_MAX, "num_blocks * num_kv_heads must be below 2^31");
  WKV_CHECK_ARG(q != nullptr && aligned16(q), "q must be non-NULL and 16-byte aligned");
  WKV_CHECK_ARG(q_stride_t >= 0 && q_stride_h >= 0 && q_stride_t % 8 == 0 && q_stride_h % 8 == 0,
                "q strides must be non-negative multiples of 8");
  WKV_CHECK_ARG(out != nullptr && aligned16(out), "out must be non-NULL and 16-byte aligned");
  WKV_CHECK_ARG(out_stride_t >= 0 && out_stride_h >= 0 && out_stride_t % 4 == 0 && out_stride_h % 4 == 0,
                "out strides must be non-negative multiples of 4");
  WKV_CHECK_ARG(cu_seqlens_q != nullptr && seq_lens != nullptr && block_table != nullptr,
                "cu_seqlens_q / seq_lens / block_table is NULL");
  WKV_CHECK_ARG(max_blocks_per_seq > 0 && bt_stride >= max_blocks_per_seq, "bad block table geometry");
  WKV_CHECK_ARG(max_query_len > 0 && max_seq_len >= 0, "max_query_len must be > 0 and max_seq_len >= 0");
  WKV_CHECK_ARG(std::isfinite(scale), "scale must be finite");
  const int max_seq = max_seq_len < max_blocks_per_seq * BS ? max_seq_len : max_blocks_per_seq * BS;
  WKV_CHECK_ARG(workgroups >= 0 && workgroups <= 65536, "workgroups must be in [0, 65536]");
  WKV_CHECK_ARG(static_cast<int64_t>(batch) * Hkv <= INT32_MAX / 8, "batch * num_kv_heads too large");
  const bool fp8 = cache->kv_dtype == WKV_KV_FP8_E4M3;
  const PrefillGrid pg = prefill_grid(batch, Hkv, G, D, fp8, max_query_len, max_seq, workgroups, workspace != nullptr);
  const int64_t need = prefill_workspace(pg, D);
  if (need > 0)
    WKV_CHECK_ARG(aligned16(workspace) && workspace_bytes >= need, "workspace too small: need %lld bytes, got %lld",
                  (long long)need, (long long)workspace_bytes);
  int64_t n_wg = (static_cast<int64_t>(pg.n_sub) + 7) / 8 * 8 * pg.n_inner;
  if (pg.W > 0) {  // (unless forced, room for a workgroup per unit group: at most 1,024 of them)
    const int64_t whole = pg.forced ? 0 : (static_cast<int64_t>(batch) * Hkv * pg.n_ug + 7) / 8 * 8;
    n_wg = whole > pg.W ? whole : pg.W;
  }
  WKV_CHECK_ARG(n_wg <= INT32_MAX, "prefill grid too large");
  rc = append();
  if (rc) return rc;
  const dim3 grid(static_cast<unsigned>(n_wg));
  auto s = static_cast<hipStream_t>(stream);
  auto kc = static_cast<const uint8_t *>(cache->k);
  auto vc = static_cast<const uint8_t *>(cache->v);
  auto qq = static_cast<const uint16_t *>(q);
  auto oo = static_cast<uint16_t *>(out);
  const float scale_log2 = scale * 1.4426950408889634f;
  const PrefillArgs args{kc, vc, cache->k_scale, cache->v_scale, qq, q_stride_t, q_stride_h, oo, out_stride_t,
                         out_stride_h, cu_seqlens_q, seq_lens, block_table, bt_stride, max_blocks_per_seq, max_seq,
                         Hkv, BS, static_cast<int>(cache->num_blocks), scale_log2, fast_div(BS), pg,
                         static_cast<float *>(workspace), sinks};
  const bool span = pg.by_U.d % 4 != 0;
#define WKV_PREFILL_S(Dv, F8, SH, SP) prefill_gqa_kernel<Dv, F8, SH, SP><<<grid, 64 * kPrefillWaves, 0, s>>>(args)
#define WKV_PREFILL(Dv, F8)                                                         \
  do {                                                                              \
    if (pg.W > 0) {                                                                 \
      if (span) WKV_PREFILL_S(Dv, F8, true, true); else WKV_PREFILL_S(Dv, F8, true, false);   \
    } else {                                                                        \
      if (span) WKV_PREFILL_S(Dv, F8, false, true); else WKV_PREFILL_S(Dv, F8, false, false); \
    }                                                                               \
  } while (0)
  if (D == 128) {
    if (fp8) WKV_PREFILL(128, true); else WKV_PREFILL(128, false);
  } else {
    if (fp8) WKV_PREFILL(64, true); else WKV_PREFILL(64, false);
  }
#undef WKV_PREFILL
#undef WKV_PREFILL_S
  WKV_CHECK_LAUNCH("paged prefill");
  if (pg.W > 0) {
    const dim3 mgrid(static_cast<unsigned>(Hkv * batch * pg.n_ug), static_cast<unsigned>(D / 32));
    if (D == 128)
      prefill_merge_kernel<128><<<mgrid, 64 * kPrefillWaves, 0, s>>>(static_cast<float *>(workspace), oo,
                                                                     out_stride_t, out_stride_h, cu_seqlens_q, seq_lens,
                                                                     max_seq, Hkv, pg, sinks);
    else
      prefill_merge_kernel<64><<<mgrid, 64 * kPrefillWaves, 0, s>>>(static_cast<float *>(workspace), oo,
                                                                    out_stride_t, out_stride_h, cu_seqlens_q, seq_lens,
                                                                    max_seq, Hkv, pg, sinks);
    WKV_CHECK_LAUNCH("paged prefill merge");
  }
  return WKV_OK;
}

extern "C" int wkv_prefill_gqa(const wkv_cache_t *cache, const void *key, int64_t key_stride_t, int64_t key_stride_h,
                               const void *value, int64_t value_stride_t, int64_t value_stride_h,
                               const int64_t *slot_mapping, int64_t num_tokens, const void *q, int64_t q_stride_t,
                               int64_t q_stride_h, void *out, int64_t out_stride_t, int64_t out_stride_h,
                               int32_t num_q_heads, const int32_t *cu_seqlens_q, const int32_t *seq_lens,
                               const int32_t *block_table, int64_t bt_stride, int32_t max_blocks_per_seq,
                               int32_t batch, int32_t max_query_len, int32_t max_seq_len, float scale, void *stream) {
  return launch_prefill(cache, key, key_stride_t, key_stride_h, value, value_stride_t, value_stride_h, slot_mapping,
                        num_tokens, q, q_stride_t, q_stride_h, out, out_stride_t, out_stride_h, num_q_heads,
                        cu_seqlens_q, seq_lens, block_table, bt_stride, max_blocks_per_seq, batch, max_query_len,
                        max_seq_len, scale, 0, nullptr, 0, nullptr, stream);
}

extern "C" int wkv_prefill_gqa_sinks(const wkv_cache_t *cache, const void *key, int64_t key_stride_t,
                                     int64_t key_stride_h, const void *value, int64_t value_stride_t,
                                     int64_t value_stride_h, const int64_t *slot_mapping, int64_t num_tokens,
                                     const void *q, int64_t q_stride_t, int64_t q_stride_h, void *out,
                                     int64_t out_stride_t, int64_t out_stride_h, int32_t num_q_heads,
                                     const int32_t *cu_seqlens_q, const int32_t *seq_lens,
                                     const int32_t *block_table, int64_t bt_stride, int32_t max_blocks_per_seq,
                                     int32_t batch, int32_t max_query_len, int32_t max_seq_len, float scale,
                                     const float *sinks, void *stream) {
  WKV_CHECK_ARG(sinks != nullptr && reinterpret_cast<uintptr_t>(sinks) % 4 == 0, "sinks must be non-NULL fp32");
  return launch_prefill(cache, key, key_stride_t, key_stride_h, value, value_stride_t, value_stride_h, slot_mapping,
                        num_tokens, q, q_stride_t, q_stride_h, out, out_stride_t, out_stride_h, num_q_heads,
                        cu_seqlens_q, seq_lens, block_table, bt_stride, max_blocks_per_seq, batch, max_query_len,
                        max_seq_len, scale, 0, nullptr, 0, sinks, stream);
}

extern "C" int64_t wkv_prefill_workspace_size(int32_t batch, int32_t kv_dtype, int32_t num_kv_heads,
                                              int32_t num_q_heads, int32_t head_dim, int32_t max_query_len,
                                              int32_t max_seq_len, int32_t workgroups) {
  if (batch < 0 || batch > 65535 || num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads != 0 ||
      head_dim <= 0 || max_query_len < 0 || max_seq_len < 0 || workgroups < 0 || workgroups > 65536)
    return -1;
  if (batch == 0 || max_query_len == 0 || static_cast<int64_t>(batch) * num_kv_heads > INT32_MAX / 8) return 0;
  return prefill_workspace(prefill_grid(batch, num_kv_heads, num_q_heads / num_kv_heads, head_dim,
                                        kv_dtype == WKV_KV_FP8_E4M3, max_query_len, max_seq_len, workgroups, true),
                           head_dim);
}

extern "C" int wkv_prefill_gqa_shared(const wkv_cache_t *cache, const void *key, int64_t key_stride_t,
                                     int64_t key_stride_h, const void *value, int64_t value_stride_t,
                                     int64_t value_stride_h, const int64_t *slot_mapping, int64_t num_tokens,
                                     const void *q, int64_t q_stride_t, int64_t q_stride_h, void *out,
                                     int64_t out_stride_t, int64_t out_stride_h, int32_t num_q_heads,
                                     const int32_t *cu_seqlens_q, const int32_t *seq_lens,
                                     const int32_t *block_table, int64_t bt_stride, int32_t max_blocks_per_seq,
                                     int32_t batch, int32_t max_query_len, int32_t max_seq_len, float scale,
                                     int32_t workgroups, void *workspace, int64_t workspace_bytes,
                                     const float *sinks, void *stream) {
  WKV_CHECK_ARG(reinterpret_cast<uintptr_t>(sinks) % 4 == 0, "sinks must be fp32");
  return launch_prefill(cache, key, key_stride_t, key_stride_h, value, value_stride_t, value_stride_h, slot_mapping,
                        num_tokens, q, q_stride_t, q_stride_h, out, out_stride_t, out_stride_h, num_q_heads,
                        cu_seqlens_q, seq_lens, block_table, bt_stride, max_blocks_per_seq, batch, max_query_len,
                        max_seq_len, scale, workgroups, workspace, workspace_bytes, sinks, stream);
}
