// Shared helpers of the sequence-mixer kernels (libumbrella_seq.so): a third storage policy (fp32) beside the 16-bit ones
// of common.h, typed element access, and the paged key/value addressing.
#pragma once
#include "common.h"
#include "../../include/umbrella_seq.h"

struct F32 {};

template <typename P> struct El { typedef u16 type; };
template <> struct El<F32> { typedef float type; };

template <typename P> __device__ __forceinline__ float ldf(const typename El<P>::type* p) { return P::to_f(*p); }
template <> __device__ __forceinline__ float ldf<F32>(const float* p) { return *p; }
template <typename P> __device__ __forceinline__ void stf(typename El<P>::type* p, float v) { *p = P::from_f(v); }
template <> __device__ __forceinline__ void stf<F32>(float* p, float v) { *p = v; }

#define DISPATCH_SEQ_DTYPE(dt, ...)                          \
  if ((dt) == UMB_SEQ_BF16) { using P = BF16; __VA_ARGS__ }  \
  else if ((dt) == UMB_SEQ_F16) { using P = F16; __VA_ARGS__ } \
  else if ((dt) == UMB_SEQ_F32) { using P = F32; __VA_ARGS__ } \
  else return UMB_EINVAL;

static inline size_t seq_elem_bytes(int dt) { return dt == UMB_SEQ_F32 ? 4 : 2; }

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + __expf(-x)); }
// log(sigmoid(x)) without overflow on either side
__device__ __forceinline__ float log_sigmoidf_(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }
// z / (1 + e^-u) as exactly as expf and a division give it, in two thirds of their instructions: e^-u as a power of two, its exponent taken apart
// into a whole number and a rest (Cody and Waite; v_exp_f32 on the rest), and one step on the quotient.  Numerator and denominator are a quarter of
// what they are, so that the reciprocal of a denominator of up to 2^128 is none that v_rcp_f32 flushes to zero; beyond it e^-u is infinite and the
// quotient 0, as there.  Infinities and NaN of z as there (the step is dropped where it is not a number).  A NaN of u alone is lost in its bounds:
// gated_ below is for a u that z does not follow from.
// Error of z = u against 64 bits, in 2^-24 of the value, over |u| < 30 / -88.7 < u < -87.2: largest 3.04 / 2.01, root mean square 0.582 / 0.604,
// all as there.  A prompt's gated feed-forward does 64 of these a lane behind its products (16384 x 2048, 2048 tokens: 125 us -> 111 with them, the
// biases and the choice of the epilogue out of the loop over tokens).
__device__ __forceinline__ float over_one_plus_exp(float z, float u) {
#pragma clang fp contract(off)
  const float c = __builtin_amdgcn_fmed3f(u, -110.f, 110.f), h = -c * 1.44269502f, n = __builtin_rintf(h);
  const float l = fmaf(-c, 1.92596303e-8f, fmaf(-c, 1.44269502f, -h));         // log2(e) in two parts
  const float d = fmaf(__builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((h - n) + l), (int)n), 0.25f, 0.25f), t = 0.25f * z;
  const float r = __builtin_amdgcn_rcpf(d), q = t * r, p = fmaf(fmaf(-q, d, t), r, q);
  return p == p ? p : q;
}
__device__ __forceinline__ float siluf_(float x) { return over_one_plus_exp(x, x); }
__device__ __forceinline__ float gated_(float z, float u) { const float y = over_one_plus_exp(z, u); return u == u ? y : u; }

// ---- paged key/value store: element offsets (in elements) of one token's / one pooled block's D-vector
__device__ __forceinline__ long pkv_tok(const UmbPagedKV& kv, int slot, int pos, int g, int G, int D) {
  const int pg = kv.pages[(long)slot * kv.max_pages + pos / kv.page];
  return (((long)pg * G + g) * kv.page + pos % kv.page) * D;
}
__device__ __forceinline__ long pkv_blk(const UmbPagedKV& kv, int slot, int b, int pool, int g, int G, int D) {
  const int e = b * pool + pool - 1;                      // the block's last position
  const int pg = kv.pages[(long)slot * kv.max_pages + e / kv.page];
  const int npb = (kv.page + pool - 1) / pool;
  return (((long)pg * G + g) * npb + (e % kv.page) / pool) * D;
}

// Dynamic LDS above the default limit needs the function attribute.  It is set once per kernel and size (a function-local
// static per kernel instantiation), i.e. by the first eager launch: a step that is being captured into a hipGraph has run
// eagerly before and makes no such call.
template <auto Kernel> static inline int ensure_dynamic_lds(size_t bytes) {
  static size_t granted = 48 * 1024;
  if (bytes > granted) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
      return UMB_EHIP;
    granted = bytes;
  }
  return UMB_OK;
}

// ---- rows walked in quads (seq_norm.hip, seq_hyper.hip): four elements in one load of 16 bytes, or of 8 from 16-bit storage
template <typename P> __device__ __forceinline__ f32x4 ld4(const typename El<P>::type* p) {
  if constexpr (sizeof(typename El<P>::type) == 4) return *reinterpret_cast<const f32x4*>(p);
  else {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p);
    return f32x4{lo_f<P>(v[0]), hi_f<P>(v[0]), lo_f<P>(v[1]), hi_f<P>(v[1])};
  }
}
template <typename P> __device__ __forceinline__ void st4(typename El<P>::type* p, f32x4 v) {
  if constexpr (sizeof(typename El<P>::type) == 4) *reinterpret_cast<f32x4*>(p) = v;
  else *reinterpret_cast<u32x2*>(p) = u32x2{pack2<P>(v[0], v[1]), pack2<P>(v[2], v[3])};
}
// A sublayer's output may stand in `parts` slabs (at most PARTS_MAX, `slab` floats apart) of partial sums: a product whose K was split.
// y holds this thread's quads of slab 0; the others' are added in order, their loads all in flight.
constexpr int PARTS_MAX = 4;
template <int NE, typename Off> __device__ __forceinline__ void add_parts(f32x4 (&y)[NE], const float* __restrict__ src, int parts, long slab, Off off) {
  if (parts == 1) return;                            // (the other output of a pair)
  f32x4 a[NE], b[NE], c[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const float* p = src + off(e) + slab;
    a[e] = *reinterpret_cast<const f32x4*>(p);
    if (parts > 2) b[e] = *reinterpret_cast<const f32x4*>(p + slab);
    if (parts > 3) c[e] = *reinterpret_cast<const f32x4*>(p + 2 * slab);
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    y[e] += a[e];
    if (parts > 2) y[e] += b[e];
    if (parts > 3) y[e] += c[e];
  }
}
__device__ __forceinline__ float sq4(f32x4 v) { return v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]; }

// One residual stream's write, mx x + ot (m y), by kernels with NE quads a thread.  The order of the two roundings is written down, and not the same in both:
// the first product is rounded by itself where a thread has one quad (few rows, and those of up to 1024 elements; the products that form a seam's rows among
// them), the second where it has several (from QUAD_ROWS rows on, and beyond 4096 elements).  A longer step's residual may so differ from a shorter one's in its
// last bit.
template <int NE> __device__ __forceinline__ f32x4 stream_write(float mx, f32x4 x, float ot, float m, f32x4 y) {
  f32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = NE == 1 ? fmaf(ot, m * y[e], mx * x[e]) : fmaf(mx, x[e], ot * (m * y[e]));
  return r;
}
// and of two outputs side by side, a fa wa + b fb wb
template <int NE> __device__ __forceinline__ f32x4 pair_sum(f32x4 a, float fa, f32x4 wa, f32x4 b, float fb, f32x4 wb) {
  f32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = NE == 1 ? fmaf(b[e] * fb, wb[e], a[e] * fa * wa[e]) : fmaf(a[e] * fa, wa[e], b[e] * fb * wb[e]);
  return r;
}
// block_sum of a row's squares with the waves' sums added in pairs: with 16 of them one after the other the scale of a row of 4096 was off by
// 0.795 x 2^-24 in the mean (root mean square), in pairs by 0.698 -- as good as four waves with more elements each
template <int NT> __device__ __forceinline__ float row_sum(float v, float* red /* >= NT / 64 floats of LDS */) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t[NT / 64];
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) t[i] = red[i];
#pragma unroll
  for (int m = NT / 128; m >= 1; m >>= 1)
#pragma unroll
    for (int i = 0; i < m; ++i) t[i] += t[i + m];
  return t[0];
}

// whether a (row, group) can be walked in quads (the rows of every operand 16 bytes apart and aligned; 16-bit ones 8)
static inline bool quads_ok(int W, int groups, const void* a, const void* b = nullptr, const void* c = nullptr, const void* d = nullptr,
                            const void* e = nullptr, const void* f = nullptr, const void* g = nullptr) {
  const int gs = W / groups;
  return gs % 4 == 0 && gs <= 8192 && groups <= 65535 &&
         ((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d | (uintptr_t)e | (uintptr_t)f | (uintptr_t)g) % 16 == 0;
}
// Groups of at most 64 elements leave three quarters of a wave idle, which shows once there are a few workgroups per unit: a wave per group
// there (2000 x 3 x 64: embedding 3.3 us, 3.7 in quads, final norm 3.1 / 3.4)
static inline bool quads_fill(int gs, long rows) { return gs > 64 || rows < 1024; }
// Rows beyond 1024 elements: one quad a thread where rows are few; from 400 rows on the chip is full either way and two or four quads a thread let
// several rows share a compute unit, one's loads behind another's sums (us, 4-byte elements by 256 threads / one quad / these: pair seam
// 700 x 3072 10.0 / 11.4 / 8.6, seam 2000 x 4096 27.5 / 21.1 / 19.7, one-stream seam 2000 x 4096 19.3 / 20.4 / 19.6, embedding 2000 x 3072 11.5 /
// 12.9 / 11.4; 256 rows: one quad is ahead or equal).
constexpr long QUAD_ROWS = 400;
#define BY_QUADS(gs, rows, LAUNCH)        \
  do {                                    \
    if ((gs) <= 256) LAUNCH(64, 1);       \
    else if ((gs) <= 512) LAUNCH(128, 1); \
    else if ((gs) <= 1024) LAUNCH(256, 1); \
    else if ((rows) >= QUAD_ROWS) {       \
      if ((gs) <= 2048) LAUNCH(256, 2);   \
      else if ((gs) <= 4096) LAUNCH(256, 4); \
      else LAUNCH(512, 4);                \
    } else if ((gs) <= 2048) LAUNCH(512, 1); \
    else if ((gs) <= 4096) LAUNCH(1024, 1); \
    else LAUNCH(1024, 2);                 \
  } while (0)

// Columns a thread of the token-by-token scan (seq_gla.hip).  A token's decays, keys and queries are read from LDS once for all of a thread's
// columns, and those reads are the time where the rows of all stretches fill the chip; where the longest stretch's walk is the time, more columns make
// its steps longer.  The line: workgroups of 16 columns that the rows keep busy over that walk, times rows a lane (keys / 16).  us with 1 / 2 / 4 columns,
// heads x keys x values: 16 x 128 x 256, one stretch of 96 36 / 44 / 61, 2 41 / 46 / 61, 4 74 / 51 / 64, 8 116 / 93 / 70, 16 of 51 - 96 184 / 133 / 117; 8 x 256 x 256, 2
// of 100 66 / 80 / 113, 8 252 / 158 / 116; 32 x 64 x 64, 8 of 100 39 / 39 / 46, 32 113 / 92 / 92.  max_len 0: nothing is known of the stretches, one column.
static inline int lin_scan_cols(int T, int max_len, int H, int D, int Dv) {
  const int nr = (D + 15) / 16;
  if (max_len < 1) return 1;
  const double busy = (double)T / max_len * H * ((Dv + 15) / 16) * nr;
  return nr % 4 ? 1 : busy >= 16384 ? 4 : busy >= 8192 ? 2 : 1;
}
