// Attention of single tokens (16-bit storage, key size a multiple of 32, value size 64, 128 or 256, latents also 512): what the decode kernels of
// seq_battn.hip and seq_pwattn.hip share.
//
// A wave takes ROUNDS of 16 keys.  Scores: lane (key lane % 16, quarter lane / 16) holds every fourth 16-byte piece of its key's row, so
// one load instruction reads 64 contiguous bytes of 16 rows and a whole round is D / 32 of them; the quarters are added by lane swaps.
// Values: LPR = E / 8 lanes hold one row in 16-byte pieces, 64 / LPR rows per load instruction; a lane keeps 8 columns per query row and
// the row groups are added once, after the last round.  The value rows do not wait for the scores: all of a round's loads are in flight
// together, and the page-table entry of the next round with them.
//
// What bounds it is latency, not bytes.  A round of 64 keys (a key per lane, a value column per lane, eight rows in flight) gave 64 keys to
// ONE wave as ten dependent memory trips while the other fifteen waves of its workgroup were idle: 19 to 23 us at 40 keys.
#pragma once
#include "seq_common.h"
#include <type_traits>

// a = {a.lo, b.lo}, b = {a.hi, b.hi} in halves of 32 lanes / in rows of 16 lanes, pairwise.  Written out: the builtin's second result came
// back as its first.  Volatile: not to be moved under a narrower execution mask.
__device__ __forceinline__ void swap32(float& a, float& b) { asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ void swap16(float& a, float& b) { asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
template <int N> __device__ __forceinline__ float ror16(float v) {            // rotated by N lanes inside its row of 16
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xf, 0xf, false));
}
__device__ __forceinline__ float row_max16(float v) {
  v = fmaxf(v, ror16<8>(v));
  v = fmaxf(v, ror16<4>(v));
  v = fmaxf(v, ror16<2>(v));
  return fmaxf(v, ror16<1>(v));
}
__device__ __forceinline__ float row_add16(float v) {
  v += ror16<8>(v);
  v += ror16<4>(v);
  v += ror16<2>(v);
  return v + ror16<1>(v);
}
// sum over the four rows of 16 lanes, in every lane
__device__ __forceinline__ float add_rows(float v) {
  float a = v, b = v;
  swap32(a, b);
  a += b;
  b = a;
  swap16(a, b);
  return a + b;
}

// Sum of squares of a row of 64, 128 or 256 that D / 4 neighbouring lanes hold in quads, in every lane of them.  The order is that of a wave with an element a lane:
// those 64 apart, one after the other (LAST_FIRST: the last rounded first), then those 32, 16, .. 1 apart; a row is scaled by the same bits whichever kernel
// prepares it.  (fmaf with 0: a product alone would be contracted into the sum behind it.)
template <int D, bool LAST_FIRST> __device__ __forceinline__ float quads_square(f32x4 x) {
  float s[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (D == 64) s[k] = fmaf(x[k], x[k], 0.f);
    else if constexpr (D == 128) {
      float a = x[k], b = x[k];
      swap16(a, b);
      s[k] = LAST_FIRST ? fmaf(a, a, fmaf(b, b, 0.f)) : fmaf(b, b, fmaf(a, a, 0.f));
    } else {
      static_assert(D == 256 && !LAST_FIRST);
      float a = x[k], c = x[k];
      swap32(a, c);
      float b = a, d = c;
      swap16(a, b);
      swap16(c, d);
      s[k] = fmaf(d, d, fmaf(c, c, fmaf(b, b, fmaf(a, a, 0.f))));
    }
    s[k] = row_add16(s[k]);
  }
  return (s[0] + s[2]) + (s[1] + s[3]);
}
// a b + c d, both products rounded
__device__ __forceinline__ float two_products(float a, float b, float c, float d) {
#pragma clang fp contract(off)
  return a * b + c * d;
}

// The same values in 16 bits either way of rounding, whatever the compiler would make of a product in front of a conversion.  fp16: the product rounded to fp32
// first (opaque, so that it is), or once, as v_fma_mixlo_f16 does; bf16 has no such instruction.
__device__ __forceinline__ f32x4 rounded(f32x4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) asm("" : "+v"(v[i]));
  return v;
}
template <typename P> __device__ __forceinline__ u16 product_once(float a, float b) {
  if constexpr (std::is_same<P, F16>::value) {
    unsigned r;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
    return (u16)r;
  } else return P::from_f(a * b);
}

// row number of a token's / a pooled block's vectors in the paged store
__device__ __forceinline__ unsigned pkv_tok_row(const UmbPagedKV& kv, int slot, int pos, int g, int G) {
  const int pg = kv.pages[(long)slot * kv.max_pages + pos / kv.page];
  return ((unsigned)pg * G + g) * kv.page + pos % kv.page;
}
__device__ __forceinline__ unsigned pkv_blk_row(const UmbPagedKV& kv, int slot, int b, int pool, int g, int G) {
  const int e = b * pool + pool - 1;
  const int pg = kv.pages[(long)slot * kv.max_pages + e / kv.page];
  return ((unsigned)pg * G + g) * ((kv.page + pool - 1) / pool) + (e % kv.page) / pool;
}

// eight features of a row in 16 bytes of 16-bit storage, or in 32 of fp32
template <typename P> __device__ __forceinline__ void unpack8(u32x4 v, float* f) {
#pragma unroll
  for (int e = 0; e < 4; ++e) { f[2 * e] = lo_f<P>(v[e]); f[2 * e + 1] = hi_f<P>(v[e]); }
}

// partial sums of a wave: acc[N] per lane, N = 8 rows, over the 64 / LPR row groups; written to dst[row][E]
template <int RH, int LPR> __device__ __forceinline__ void store_groups(float* dst, float (&acc)[RH * 8], int lane) {
  constexpr int E = LPR * 8, N = RH * 8;
  if constexpr (LPR == 64) {                                 // a row a load: every lane has its columns' sums
#pragma unroll
    for (int v = 0; v < N; ++v) dst[(v >> 3) * E + lane * 8 + (v & 7)] = acc[v];
    return;
  }
#pragma unroll
  for (int k = 0; k < N / 2; ++k) {                          // after this register k holds value 2 k + (lane / 32)
    float a = acc[2 * k], b = acc[2 * k + 1];
    swap32(a, b);
    acc[k] = a + b;
  }
  const int b5 = lane >> 5, b4 = (lane >> 4) & 1;
  if constexpr (LPR == 32) {
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      const int v = 2 * k + b5;
      dst[(v >> 3) * E + (lane & 31) * 8 + (v & 7)] = acc[k];
    }
  } else {
#pragma unroll
    for (int k = 0; k < N / 4; ++k) {                        // and register k value 4 k + 2 (lane / 16 % 2) + lane / 32
      float a = acc[2 * k], b = acc[2 * k + 1];
      swap16(a, b);
      float s = a + b;
      if constexpr (LPR == 8) s += ror16<8>(s);
      const int v = 4 * k + 2 * b4 + b5;
      if (LPR == 16 || (lane & 8) == 0) dst[(v >> 3) * E + (lane & (LPR - 1)) * 8 + (v & 7)] = s;
    }
  }
}

static inline bool decode_rows_ok(int D, int E, int dtype, const UmbPagedKV* kv) {
  return dtype != UMB_SEQ_F32 && D % 32 == 0 && D <= 512 && (E == 64 || E == 128 || E == 256) &&
         ((uintptr_t)kv->k | (uintptr_t)kv->v | (uintptr_t)kv->kp | (uintptr_t)kv->vp) % 16 == 0;
}
