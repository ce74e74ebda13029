// Device-side fp8 append shared by the append kernel and the fused append +
// decode kernel (one wave appends one run of one KV head).
#pragma once

#include "wkv_common.h"

namespace wkv {

// ---------------------------------------------------------------------------
// Where element d of the token at offset off lies in the K and V codes.
template <int D>
__device__ __forceinline__ int64_t fp8_k_index(int64_t blk, int h, int H, int BS, int off, int d) {
  return (((blk * H + h) * (D / 16) + (d >> 4)) * BS + off) * 16 + (d & 15);
}
template <int D>
__device__ __forceinline__ int64_t fp8_v_index(int64_t blk, int h, int H, int BS, int off, int d) {
  return ((blk * H + h) * D + d) * BS + off;
}

// Four e4m3 codes times `ratio`, a power of two below 1, by the hardware
// conversions: code by code e4m3_encode(e4m3_decode(c) * ratio) (the products
// are bf16 values, for which the two encoders agree bit for bit). NaN codes
// are kept as they are, as the encoder keeps them.
__device__ __forceinline__ uint32_t fp8x4_rescale(uint32_t c, float ratio) {
  const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(c), false);
  const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(c), true);
  int r = __builtin_amdgcn_cvt_pk_fp8_f32(lo[0] * ratio, lo[1] * ratio, 0, false);
  r = __builtin_amdgcn_cvt_pk_fp8_f32(hi[0] * ratio, hi[1] * ratio, r, true);
  const uint32_t nan = ((((c & 0x7f7f7f7fu) + 0x01010101u) & 0x80808080u) >> 7) * 0xffu;  // bytes of code 0x7f or 0xff
  return (static_cast<uint32_t>(r) & ~nan) | (c & nan);
}

// Re-encodes the codes at offsets [0, first) of the (blk, h) region of K (IS_V
// false) or V at a grown scale: each code times `ratio`, an exact power of two
// below 1 (e4m3_encode(e4m3_decode(c) * ratio), code by code, as the oracle
// states it). The region is walked in 16-byte pieces, four per lane a pass,
// every load of a pass issued before its stores (a byte loop waits one memory
// round trip per byte). K [D/16][BS][16]: piece p holds token p % BS's 16
// d-values of one chunk; V [D][BS]: piece p holds tokens 16 (p % (BS/16)) ..
// + 15 of one d row. Pieces at or past `first` are not stored.
// LEAN: nothing that depends on the lane is held across a caller's loop over
// runs (the registers it saves there are worth more than forming it again).
template <int D, bool IS_V, bool LEAN = false>
__device__ __forceinline__ void fp8_reencode_block(uint8_t *__restrict__ cache, int64_t blk, int h, int H, int BS,
                                                   int first, float ratio) {
  int lane = threadIdx.x & 63;
  if constexpr (LEAN) asm volatile("" : "+v"(lane));
  u32x4 *base = reinterpret_cast<u32x4 *>(cache + (blk * H + h) * static_cast<int64_t>(D) * BS);
  const int np = D * BS / 16;
  constexpr int PL = 4;
  for (int p0 = 0; p0 < np; p0 += 64 * PL) {
    u32x4 w[PL];
#pragma unroll
    for (int k = 0; k < PL; ++k) {
      const int p = p0 + 64 * k + lane;
      if (p < np) w[k] = base[p];
    }
#pragma unroll
    for (int k = 0; k < PL; ++k) {
      const int p = p0 + 64 * k + lane;
      const int tok0 = IS_V ? 16 * (p % (BS / 16)) : p % BS;
      if (p >= np || tok0 >= first) continue;
      u32x4 o = w[k];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // the bytes of this word before `first`: all of them (K: a piece is one token)
        const int n = IS_V ? first - (tok0 + 4 * j) : 4;
        const uint32_t m = n >= 4 ? 0xffffffffu : (n <= 0 ? 0u : (1u << (8 * n)) - 1u);
        o[j] = (o[j] & ~m) | (fp8x4_rescale(o[j], ratio) & m);
      }
      base[p] = o;
    }
  }
}

// The step token's K and V rows of one head as loaded (bf16 bits, d = lane +
// 64 i): loaded apart from the rest of the append so that a caller can issue
// them early and let their round trip overlap its own start (nothing here
// waits for them; the append below converts them).
template <int D>
struct Fp8TokenRows {
  uint32_t k[D / 64], v[D / 64];
};
template <int D>
__device__ __forceinline__ void fp8_token_rows_load(Fp8TokenRows<D> &r, const uint16_t *__restrict__ krow,
                                                    const uint16_t *__restrict__ vrow) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < D / 64; ++i) {
    r.k[i] = krow[lane + 64 * i];
    r.v[i] = vrow[lane + 64 * i];
  }
}

// The step token's codes and the block's scales after its append, without
// writing anything: the same scale decision as fp8_append_token_kv (the
// token's power-of-two scale, or the block's own if that is not smaller),
// `grow` when the block's earlier codes would need re-encoding, and the
// token's K and V codes at the resulting scales, d = lane + 64 i.
template <int D>
struct Fp8TokenCodes {
  uint32_t k[D / 64], v[D / 64];
  float sk, sv;
  bool grow;
};
template <int D>
__device__ __forceinline__ Fp8TokenCodes<D> fp8_token_codes(const float *__restrict__ ks, const float *__restrict__ vs,
                                                            const Fp8TokenRows<D> &rows, int64_t blk, int off, int h,
                                                            int H) {
  constexpr int PER = D / 64;
  float xk[PER], xv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    xk[i] = bf16_bits_to_f32(static_cast<uint16_t>(rows.k[i]));
    xv[i] = bf16_bits_to_f32(static_cast<uint16_t>(rows.v[i]));
  }
  const int64_t si = blk * H + h;
  const float sk_old = off != 0 ? ks[si] : 0.f, sv_old = off != 0 ? vs[si] : 0.f;
  float ak = 0.f, av = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    ak = fmaxf(ak, fabsf(xk[i]));
    av = fmaxf(av, fabsf(xv[i]));
  }
  ak = wave_max(ak);
  av = wave_max(av);
  Fp8TokenCodes<D> c;
  c.sk = pow2_scale(ak);
  c.sv = pow2_scale(av);
  c.grow = false;
  if (off != 0) {
    c.grow = c.sk > sk_old || c.sv > sv_old;
    if (!(c.sk > sk_old)) c.sk = sk_old;
    if (!(c.sv > sv_old)) c.sv = sv_old;
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    c.k[i] = e4m3_quantize(xk[i], c.sk);
    c.v[i] = e4m3_quantize(xv[i], c.sv);
  }
  return c;
}

// fp8 append of one token (the fused decode's step token, a run of one token)
// for one head, K and V together, from its loaded rows: both old scales are
// loaded at once and both rows reduced side by side, so the two appends cost
// one chain of memory round trips instead of two. The same codes, scales and
// re-encodes as fp8_append_run_kv with a run of one token. PIECES: re-encodes
// by fp8_reencode_block, else byte by byte: with the former in the fused decode
// kernel that inlines this, a launch measured 3-4% slower even in steps where
// no block grows (fp8 Qwen2.5-7B groups and Qwen3-4B shapes, in-process A/B).
template <int D, bool PIECES = false>
__device__ __forceinline__ void fp8_append_token_kv(uint8_t *__restrict__ kc, uint8_t *__restrict__ vc,
                                                    float *__restrict__ ks, float *__restrict__ vs,
                                                    const Fp8TokenRows<D> &rows, int64_t blk, int off, int h, int H,
                                                    int BS) {
  constexpr int PER = D / 64;  // elements of a row per lane: d = lane + 64 i
  const int lane = threadIdx.x & 63;
  float xk[PER], xv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    xk[i] = bf16_bits_to_f32(static_cast<uint16_t>(rows.k[i]));
    xv[i] = bf16_bits_to_f32(static_cast<uint16_t>(rows.v[i]));
  }
  const int64_t si = blk * H + h;
  const float sk_old = off != 0 ? ks[si] : 0.f, sv_old = off != 0 ? vs[si] : 0.f;
  float ak = 0.f, av = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    ak = fmaxf(ak, fabsf(xk[i]));
    av = fmaxf(av, fabsf(xv[i]));
  }
  ak = wave_max(ak);
  av = wave_max(av);
  float sk = pow2_scale(ak), sv = pow2_scale(av);
  if (off != 0) {
    if (sk > sk_old) {  // the block's earlier K codes at the grown scale
      const float ratio = sk_old / sk;
      if constexpr (PIECES)
        fp8_reencode_block<D, false>(kc, blk, h, H, BS, off, ratio);
      else
      for (int e = lane; e < off * D; e += 64) {
        const int64_t a = fp8_k_index<D>(blk, h, H, BS, e / D, e % D);
        kc[a] = static_cast<uint8_t>(e4m3_encode(e4m3_decode(kc[a]) * ratio));
      }
    } else {
      sk = sk_old;
    }
    if (sv > sv_old) {
      const float ratio = sv_old / sv;
      if constexpr (PIECES)
        fp8_reencode_block<D, true>(vc, blk, h, H, BS, off, ratio);
      else
      for (int e = lane; e < off * D; e += 64) {
        const int64_t a = fp8_v_index<D>(blk, h, H, BS, e / D, e % D);
        vc[a] = static_cast<uint8_t>(e4m3_encode(e4m3_decode(vc[a]) * ratio));
      }
    } else {
      sv = sv_old;
    }
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    kc[fp8_k_index<D>(blk, h, H, BS, off, lane + 64 * i)] = static_cast<uint8_t>(e4m3_quantize(xk[i], sk));
    vc[fp8_v_index<D>(blk, h, H, BS, off, lane + 64 * i)] = static_cast<uint8_t>(e4m3_quantize(xv[i], sv));
  }
  if (lane == 0) {
    ks[si] = sk;
    vs[si] = sv;
  }
}

// Codes of a and b (after the clamp to +-448; never NaN here) in bytes
// 2 w, 2 w + 1 of `old`, by the hardware conversion: for every finite input
// bit-identical to e4m3_encode (checked on the GPU for all bf16 patterns at
// several scales). NaN is the one difference -- the hardware codes +NaN 0xFF
// where e4m3_encode gives 0x7F -- so callers keep NaN off this path.
template <bool W1>
__device__ __forceinline__ uint32_t e4m3_pack2(float a, float b, uint32_t old) {
  return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(a, b, static_cast<int>(old), W1));
}

// Four bf16 pairs (words w0..w3, low half first) times inv, clamped, as 8 codes
// in two words.
__device__ __forceinline__ u32x2 e4m3_pack8(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, float inv) {
  auto lo = [&](uint32_t w) { return __builtin_amdgcn_fmed3f(__uint_as_float(w << 16) * inv, -448.f, 448.f); };
  auto hi = [&](uint32_t w) { return __builtin_amdgcn_fmed3f(__uint_as_float(w & 0xffff0000u) * inv, -448.f, 448.f); };
  u32x2 r;
  r[0] = e4m3_pack2<true>(lo(w1), hi(w1), e4m3_pack2<false>(lo(w0), hi(w0), 0u));
  r[1] = e4m3_pack2<true>(lo(w3), hi(w3), e4m3_pack2<false>(lo(w2), hi(w2), 0u));
  return r;
}

// fp8 append of one run (tokens t..t+r-1, all in block blk, the first at offset
// `first`) for one head, K and V together, by one wave: scale update, re-encode
// of the block's earlier entries when a scale grows, then the run's codes
// (e4m3_quantize's). Bound by memory round trips, so the run goes in
// pieces of 16 tokens whose rows, slots and old scales are all requested before
// the first is used (K: lane l holds token l % 16, 16-d chunks l / 16 + 4 j; V:
// RV = D / 64 rows of every token), and a run of one piece -- any run of a
// 16-token block -- stays in registers between its maximum and its codes; a
// longer run reads its pieces twice. Loads of tokens past the run repeat its
// last token (no effect on the maximum) and are not stored. 574 tokens in four
// ragged runs over partly filled blocks, 4 heads: 22.7 us with K and V one
// after the other and V a token at a time, 11.1 us so. Source rows 16-byte
// aligned (the host checks).
template <int D, bool LEAN>
__device__ __forceinline__ void fp8_append_run_body(uint8_t *__restrict__ kc, uint8_t *__restrict__ vc,
                                                    float *__restrict__ ks, float *__restrict__ vs,
                                                    const uint16_t *__restrict__ key, int64_t kst, int64_t ksh,
                                                    const uint16_t *__restrict__ val, int64_t vst, int64_t vsh,
                                                    const int64_t *__restrict__ slots, int64_t t, int r, int64_t blk,
                                                    int first, int h, int H, int BS) {
  constexpr int P = 16, NC = D / 64, RV = D / 64;
  int lane = threadIdx.x & 63;
  if constexpr (LEAN) asm volatile("" : "+v"(lane));
  const int m = lane & 15;
  const int64_t si = blk * H + h;
  const float sk_old = first != 0 ? ks[si] : 0.f, sv_old = first != 0 ? vs[si] : 0.f;
  u32x4 kw[NC][2];
  uint32_t vw[P];
  int off = 0;  // offset in the block of the piece's token m
  auto load = [&](int p0) __attribute__((always_inline)) {
    const int last = (r - p0 < P ? r - p0 : P) - 1;
    const int64_t tm = t + p0 + (m < last ? m : last);
    off = static_cast<int>(slots[tm] - blk * BS);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const uint16_t *p = key + tm * kst + h * ksh + 16 * ((lane >> 4) + 4 * j);
      kw[j][0] = *reinterpret_cast<const u32x4 *>(p);
      kw[j][1] = *reinterpret_cast<const u32x4 *>(p + 8);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const uint16_t *p = val + (t + p0 + (i < last ? i : last)) * vst + h * vsh + RV * lane;
      if constexpr (RV == 2)
        vw[i] = *reinterpret_cast<const uint32_t *>(p);
      else
        vw[i] = *p;
    }
  };
  // Largest magnitude bits (as bf16); a NaN counts as none, as fmaxf has it, and is remembered.
  uint32_t ka = 0u, va = 0u;
  bool nan = false;
  auto mag = [&](uint32_t a, uint32_t w) __attribute__((always_inline)) {
    const uint32_t x = w & 0x7fffu, y = (w >> 16) & 0x7fffu;
    nan = nan || x > 0x7f80u || y > 0x7f80u;
    return max(a, max(x > 0x7f80u ? 0u : x, y > 0x7f80u ? 0u : y));
  };
  for (int p0 = 0; p0 < r; p0 += P) {  // uniform
    load(p0);
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) ka = mag(ka, kw[j][q][e]);
#pragma unroll
    for (int i = 0; i < P; ++i) va = mag(va, vw[i]);
  }
  ka = wave_reduce(ka, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  va = wave_reduce(va, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  const bool any_nan = __any(nan);
  float sk = pow2_scale(__uint_as_float(ka << 16)), sv = pow2_scale(__uint_as_float(va << 16));
  if (first != 0) {  // the block's earlier codes are re-encoded at a grown scale (exact power-of-two ratio)
    if (sk > sk_old)
      fp8_reencode_block<D, false, LEAN>(kc, blk, h, H, BS, first, sk_old / sk);
    else
      sk = sk_old;
    if (sv > sv_old)
      fp8_reencode_block<D, true, LEAN>(vc, blk, h, H, BS, first, sv_old / sv);
    else
      sv = sv_old;
  }
  // exact: powers of two in [2^-42, 2^119], so x * (1 / s) and x / s round the same value
  const float ik = 1.0f / sk, iv = 1.0f / sv;
  auto q = [](uint32_t bits, float inv) {  // a NaN's code as e4m3_encode has it
    float v = __uint_as_float(bits << 16) * inv;
    v = (v != v) ? v : fminf(fmaxf(v, -448.0f), 448.0f);
    return e4m3_encode(v);
  };
  auto pack8 = [&](uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, float inv) __attribute__((always_inline)) {
    if (!any_nan) return e4m3_pack8(w0, w1, w2, w3, inv);  // uniform
    u32x2 o;
    o[0] = q(w0 & 0xffffu, inv) | (q(w0 >> 16, inv) << 8) | (q(w1 & 0xffffu, inv) << 16) | (q(w1 >> 16, inv) << 24);
    o[1] = q(w2 & 0xffffu, inv) | (q(w2 >> 16, inv) << 8) | (q(w3 & 0xffffu, inv) << 16) | (q(w3 >> 16, inv) << 24);
    return o;
  };
  for (int p0 = 0; p0 < r; p0 += P) {
    if (r > P) load(p0);
    const int n = r - p0 < P ? r - p0 : P;
    if (m < n) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const u32x2 a = pack8(kw[j][0][0], kw[j][0][1], kw[j][0][2], kw[j][0][3], ik);
        const u32x2 b = pack8(kw[j][1][0], kw[j][1][1], kw[j][1][2], kw[j][1][3], ik);
        *reinterpret_cast<u32x4 *>(kc + fp8_k_index<D>(blk, h, H, BS, off, 16 * ((lane >> 4) + 4 * j))) =
            u32x4{a[0], a[1], b[0], b[1]};
      }
    }
#pragma unroll
    for (int rr = 0; rr < RV; ++rr) {
      // row RV lane + rr: the rr-th half of every token's word, a byte per token
      uint8_t *row = vc + fp8_v_index<D>(blk, h, H, BS, 0, RV * lane + rr);
      auto pair = [&](int i) { return ((vw[i] >> (16 * rr)) & 0xffffu) | (((vw[i + 1] >> (16 * rr)) & 0xffffu) << 16); };
#pragma unroll
      for (int g = 0; g < P; g += 8) {
        if (g >= n) break;  // uniform
        const u32x2 c = pack8(pair(g), pair(g + 2), pair(g + 4), pair(g + 6), iv);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (g + i < n) row[__builtin_amdgcn_readlane(off, g + i)] = static_cast<uint8_t>(c[i >> 2] >> (8 * (i & 3)));
      }
    }
  }
  if (lane == 0) {
    ks[si] = sk;
    vs[si] = sv;
  }
}

// The same for callers without a register target: compiled on its own before it
// is inlined, it comes out 5 to 10% faster (d=64, runs of 63 tokens in blocks of 64: 19.8 us
// against 21.3) with 199 registers in the place of some 90.
template <int D>
__device__ void fp8_append_run_kv(uint8_t *__restrict__ kc, uint8_t *__restrict__ vc, float *__restrict__ ks,
                                  float *__restrict__ vs, const uint16_t *__restrict__ key, int64_t kst, int64_t ksh,
                                  const uint16_t *__restrict__ val, int64_t vst, int64_t vsh,
                                  const int64_t *__restrict__ slots, int64_t t, int r, int64_t blk, int first, int h,
                                  int H, int BS) {
  fp8_append_run_body<D, false>(kc, vc, ks, vs, key, kst, ksh, val, vst, vsh, slots, t, r, blk, first, h, H, BS);
}

// fp8 append of a whole fresh block (16 tokens t..t+15 at offsets 0..15 of
// block blk, block_size 16) for one head, K and V, by one wave -- the prompt
// case. The block starts afresh (its scale is the run's), so nothing earlier
// is re-encoded. Returns false, having written nothing, when the block's
// inputs hold a NaN (the caller then takes fp8_append_run_kv, which codes NaN
// as e4m3_encode does). K: lane l quantises token l % 16, 16-d chunks
// l / 16 + 4 j, each one 16-byte store; V: lane l owns d rows RV l .. RV l +
// RV - 1 (RV = D / 64) and stores each row's 16 tokens as 16 bytes. Each
// block's absolute maximum is an integer maximum of bf16 magnitude bits (a
// NaN's bits exceed infinity's). Source rows 16-byte aligned (the host checks).
template <int D>
__device__ bool fp8_append_block16(uint8_t *__restrict__ kc, uint8_t *__restrict__ vc, float *__restrict__ ks,
                                   float *__restrict__ vs, const uint16_t *__restrict__ key, int64_t kst,
                                   int64_t ksh, const uint16_t *__restrict__ val, int64_t vst, int64_t vsh,
                                   int64_t t, int64_t blk, int h, int H) {
  constexpr int BS = 16, NC = D / 64, RV = D / 64;
  const int lane = threadIdx.x & 63;
  const int m = lane & 15;
  u32x4 kw[NC][2];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const uint16_t *p = key + (t + m) * kst + h * ksh + 16 * ((lane >> 4) + 4 * j);
    kw[j][0] = *reinterpret_cast<const u32x4 *>(p);
    kw[j][1] = *reinterpret_cast<const u32x4 *>(p + 8);
  }
  uint32_t vw[BS];  // token i's RV values of this lane's rows (RV = 2: one word, RV = 1: the low half)
#pragma unroll
  for (int i = 0; i < BS; ++i) {
    const uint16_t *p = val + (t + i) * vst + h * vsh + RV * lane;
    if constexpr (RV == 2)
      vw[i] = *reinterpret_cast<const uint32_t *>(p);
    else
      vw[i] = *p;
  }
  uint32_t ka = 0u, va = 0u;  // largest magnitude bits, as bf16
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = kw[j][q][e];
        ka = max(ka, max(w & 0x7fffu, (w >> 16) & 0x7fffu));
      }
#pragma unroll
  for (int i = 0; i < BS; ++i) va = max(va, max(vw[i] & 0x7fffu, (vw[i] >> 16) & 0x7fffu));
  ka = wave_reduce(ka, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  va = wave_reduce(va, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  if (ka > 0x7f80u || va > 0x7f80u) return false;  // uniform: a NaN somewhere
  const float sk = pow2_scale(__uint_as_float(ka << 16)), sv = pow2_scale(__uint_as_float(va << 16));
  const float ik = 1.0f / sk, iv = 1.0f / sv;  // exact: powers of two
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const u32x2 a = e4m3_pack8(kw[j][0][0], kw[j][0][1], kw[j][0][2], kw[j][0][3], ik);
    const u32x2 b = e4m3_pack8(kw[j][1][0], kw[j][1][1], kw[j][1][2], kw[j][1][3], ik);
    *reinterpret_cast<u32x4 *>(kc + fp8_k_index<D>(blk, h, H, BS, m, 16 * ((lane >> 4) + 4 * j))) =
        u32x4{a[0], a[1], b[0], b[1]};
  }
#pragma unroll
  for (int rr = 0; rr < RV; ++rr) {
    // row RV lane + rr: the rr-th half of every token's word, 16 tokens
    auto row = [&](int i) { return (vw[i] >> (16 * rr)) & 0xffffu; };
    auto pair = [&](int i) { return row(i) | (row(i + 1) << 16); };
    const u32x2 a = e4m3_pack8(pair(0), pair(2), pair(4), pair(6), iv);
    const u32x2 b = e4m3_pack8(pair(8), pair(10), pair(12), pair(14), iv);
    const u32x4 out = {a[0], a[1], b[0], b[1]};
    *reinterpret_cast<u32x4 *>(vc + fp8_v_index<D>(blk, h, H, BS, 0, RV * lane + rr)) = out;
  }
  if (lane == 0) {
    ks[blk * H + h] = sk;
    vs[blk * H + h] = sv;
  }
  return true;
}

}  // namespace wkv
