// Causal softmax attention with a learned bias by distance, grouped query heads, over the paged key/value store.
//     q_i = unit_rms(W_q h_i) * w_q * temp(i)       k_j = unit_rms(W_k h_j) * w_k       v_j = unit_rms(W_v h_j)
//     score(i, j, h) = q_i . k_j * scale + bias[h][min(i - j, n_dist - 1)]      (j <= i, i - j < window)
//     out_i = c * sigmoid(gate_i[h]) * softmax_j(score) . v
// With softcap > 0 the scaled product is capped before the bias joins it: softcap tanh(q . k scale / softcap).
// temp(i) = 1 + coef ln(floor((i + 1) / every) + 1) sharpens the queries of long contexts; the bias table is indexed by the
// clamped distance itself (whatever bucketing a design uses is expanded into it at load).  Keys and values are cached as
// normed (storage dtype); queries, scores, weights, maxima and sums are fp32 (expf, not the fast intrinsic).
//
// The general form (umb_attn_*, UmbAttnForm) adds, each by parameter:
//   chunk   position i sees only keys of its own run of `chunk` positions, counted from position 0 of the sequence
//   sink    a per-head score that joins the softmax denominator with no key and no value
//   maps    2: differential attention -- every head has two query / key maps over the SAME values (a cached key row is [map 1 |
//           map 2]); with a1, a2 their softmax outputs o = a1 - lambda a2, and the head's o over its root mean square goes out.
//           The two maps of a head are two rows of one workgroup: the value rows are read once for both.
//   keep_first   the first keep_first positions stay visible (at their true distance) whatever the window and the chunk hide:
//           the walk over the keys takes those of them that lie before its first position in front, as one range
//   gate_elem    the output gate is a row of H E columns, one sigmoid per output element, instead of one per head
// and its prep adds rotary positions (either pair layout, a constant on cos and sin), norms by choice, queries alone (a
// layer that reads another layer's keys and values), and values mixed with those of another layer (UmbValueMix): what is cached is
// (1 - lambda) v + lambda first, with `first` the same tokens' values as an earlier layer's prep left them.
//
// prep: one wave per (token, head slot): query heads -> fp32 q, key heads -> cache K, value heads -> cache V.
// attend (vector pipe, any dtype and head size): workgroup = (token, RH query heads of ONE key/value head, so one pass over
// the keys serves them all); waves take 64-key rounds by round number; score phase lane = key, value phase lane = value
// column with eight keys' rows in flight; per-wave running maximum / denominator, merged through LDS in wave order.  Which
// keys land in which wave and round depends on the query's position and on the launch (waves an item, splits of a token's keys, prompt tiles):
// the same token in another batch, or of a prompt cut elsewhere, agrees to fp32 rounding and not bit for bit.
#include "seq_common.h"
#include <algorithm>
#include "seq_decode.h"
#include "seq_rows.h"

static inline bool bsa_kv_ok(const UmbPagedKV* kv) { return kv && kv->k && kv->v && kv->pages && kv->page >= 1 && kv->max_pages >= 1; }

// HQ = H maps query slots, GK = G maps key slots (key slot x: key/value head x / maps, map x % maps), G value slots (GV = 0: none)
struct AttnPrep {
  int HQ, GK, G, GV, D, E, maps;
  int norm_qk, norm_v;                     // unit RMS (times the weight, where there is one) of q and k; of v
  int rot_dims, layout;
  float rot_mult;
  float temp_coef;
  int temp_every;
  float eps;
  UmbValueMix mix;                         // first: values to mix in; keep: where this layer's own go (fp32 rows of G E); null: neither
};

// a wave's: one row of n values or one row of D queries or keys, put(i, value) for each.  p: the token's position, temp: on queries
__device__ __forceinline__ float attn_prep_scale(const float* __restrict__ src, int n, int norm, float eps) {
  float ss = 0.f;
  const int lane = threadIdx.x & 63;
  if (!norm) return 1.f;
  for (int i = lane; i < n; i += 64) { const float v = src[i]; ss += v * v; }
  ss = wave_sum(ss);
  return 1.f / sqrtf(ss / (float)n + eps);
}
template <typename Put>
__device__ __forceinline__ void attn_prep_value(const float* __restrict__ src, const AttnPrep& a, long o, bool keep, Put put) {
  const float f = attn_prep_scale(src, a.E, a.norm_v, a.eps);
  for (int i = threadIdx.x & 63; i < a.E; i += 64) {
    float v = src[i] * f;
    if (keep && a.mix.keep) a.mix.keep[o + i] = v;
    if (a.mix.first) v = (1.f - a.mix.lambda) * v + a.mix.lambda * a.mix.first[o + i];
    put(i, v);
  }
}
template <typename P, typename Put>
__device__ __forceinline__ void attn_prep_row(const float* __restrict__ src, const AttnPrep& a, const typename El<P>::type* __restrict__ w,
                                              const float* __restrict__ freq, int p, float temp, Put put) {
  const float f = attn_prep_scale(src, a.D, a.norm_qk, a.eps);
  const int half = a.rot_dims >> 1;
  for (int i = threadIdx.x & 63; i < a.D; i += 64) {
    float v = src[i] * f * (w ? ldf<P>(w + i) : 1.f);
    if (i < a.rot_dims) {
      int fi, other;
      bool first;
      if (a.layout == 0) { first = i < half; fi = first ? i : i - half; other = first ? i + half : i - half; }
      else { first = (i & 1) == 0; fi = i >> 1; other = i ^ 1; }
      const float u = src[other] * f * (w ? ldf<P>(w + other) : 1.f);
      float sn, cs;
      sincosf((float)p * freq[fi], &sn, &cs);
      sn *= a.rot_mult;
      cs *= a.rot_mult;
      v = first ? v * cs - u * sn : v * cs + u * sn;
    }
    put(i, v * temp);
  }
}
// The same for the decode kernels (D a multiple of 32), compact because what a launch executes once costs its fetch: a pair of features a lane, the angle
// worked out once for both, in one place for queries and keys; the operands are asked for together, in front of the norm's sum (of the same order).
template <typename P, typename Put>
__device__ __forceinline__ void attn_prep_pairs(const float* __restrict__ src, const AttnPrep& a, const typename El<P>::type* __restrict__ w,
                                                const float* __restrict__ freq, int p, float temp, Put put) {
  const int lane = threadIdx.x & 63, half = a.rot_dims >> 1, pairs = a.D >> 1;
  int i0, i1;
  float u, v, wu, wv, fr;
  auto get = [&](int m) __attribute__((always_inline)) {
    m = min(m, pairs - 1);
    const bool split = a.layout == 0 && m < half;
    i0 = split ? m : 2 * m;                                  // layout 0: pairs behind the turned ones stand at rot_dims + 2 (m - half) = 2 m too
    i1 = split ? m + half : 2 * m + 1;
    u = src[i0];
    v = src[i1];
    wu = w ? ldf<P>(w + i0) : 1.f;
    wv = w ? ldf<P>(w + i1) : 1.f;
    fr = m < half ? freq[m] : 0.f;
  };
  get(lane);
  float f = 1.f;
  if (a.norm_qk) {
    float ss = 0.f;
#pragma unroll 1
    for (int i = lane; i < a.D; i += 128) {
      const float x = src[i], y = i + 64 < a.D ? src[i + 64] : 0.f;
      ss = fmaf(y, y, fmaf(x, x, ss));
    }
    f = 1.f / sqrtf(wave_sum(ss) / (float)a.D + a.eps);
  }
#pragma unroll 1
  for (int b = 0;;) {
    const int m = b + lane;
    float x = u * f * wu, y = v * f * wv;
    if (m < half) {
      float sn, cs;
      sincosf((float)p * fr, &sn, &cs);
      sn *= a.rot_mult;
      cs *= a.rot_mult;
      const float rx = fmaf(x, cs, -(y * sn)), ry = fmaf(y, cs, x * sn);
      x = rx;
      y = ry;
    }
    if (m < pairs) {
      put(i0, x * temp);
      put(i1, y * temp);
    }
    b += 64;
    if (b >= pairs) break;
    get(b + lane);
  }
}
template <int NC, typename Put>
__device__ __forceinline__ void attn_prep_value_few(const float* __restrict__ src, const AttnPrep& a, long o, bool keep, Put put) {
  const int lane = threadIdx.x & 63;
  float v[NC], m[NC], f = 1.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    v[c] = src[lane + 64 * c];
    m[c] = a.mix.first ? a.mix.first[o + lane + 64 * c] : 0.f;
  }
  if (a.norm_v) {
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) ss = fmaf(v[c], v[c], ss);
    f = 1.f / sqrtf(wave_sum(ss) / (float)(64 * NC) + a.eps);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float x = v[c] * f;
    if (keep && a.mix.keep) a.mix.keep[o + lane + 64 * c] = x;
    if (a.mix.first) x = fmaf(1.f - a.mix.lambda, x, a.mix.lambda * m[c]);
    put(lane + 64 * c, x);
  }
}
__device__ __forceinline__ float attn_temp(const AttnPrep& a, int p) { return a.temp_every > 0 ? 1.f + a.temp_coef * logf((float)((p + 1) / a.temp_every + 1)) : 1.f; }

template <typename P>
__global__ __launch_bounds__(256) void attn_prep_kernel(float* __restrict__ q, UmbPagedKV kv, const float* __restrict__ proj, int ld,
                                                        const typename El<P>::type* __restrict__ w_q,
                                                        const typename El<P>::type* __restrict__ w_k, const int* __restrict__ pos,
                                                        const int* __restrict__ slot, const float* __restrict__ freq, int T,
                                                        AttnPrep a) {
  typedef typename El<P>::type El_;
  const int wave = threadIdx.x >> 6;
  const int per = a.HQ + a.GK + a.GV;
  const long item = (long)blockIdx.x * 4 + wave;
  if (item >= (long)T * per) return;
  const int t = (int)(item / per), hs = (int)(item % per);
  const bool is_v = hs >= a.HQ + a.GK, is_q = hs < a.HQ;
  const int D = a.D, p = pos[t];
  const float* src = proj + (long)t * ld + (is_v ? (a.HQ + a.GK) * D + (hs - a.HQ - a.GK) * a.E : hs * D);
  if (is_v) {
    const int g = hs - a.HQ - a.GK;
    El_* row = reinterpret_cast<El_*>(kv.v) + pkv_tok(kv, slot[t], p, g, a.G, a.E);
    attn_prep_value(src, a, ((long)t * a.G + g) * a.E, true, [&](int i, float v) { stf<P>(row + i, v); });
    return;
  }
  const int ks = hs - a.HQ;
  El_* krow = is_q ? nullptr : reinterpret_cast<El_*>(kv.k) + pkv_tok(kv, slot[t], p, ks / a.maps, a.G, a.maps * D) + (ks % a.maps) * D;
  float* qrow = q + ((long)t * a.HQ + (is_q ? hs : 0)) * D;
  attn_prep_row<P>(src, a, is_q ? w_q : w_k, freq, p, is_q ? attn_temp(a, p) : 1.f, [&](int i, float v) {
    if (is_q) qrow[i] = v;
    else stf<P>(krow + i, v);
  });
}

// The same for many items, rows of 64 or 128 whose turned part is whole quads: a wave takes PREP_QUADS quads a lane of one token's neighbouring rows (queries
// and keys, or values), two or four rows side by side, all loads in flight, and works the angles out once for all of them.
// Vector work bounded what it replaces (four slots a wave, an element a lane, the angles again for every four: some 250 instructions a slot, quotients and
// sines among them).  us, that / this, bf16: 2466 tokens, 32 + 8 + 8 slots of 64 33.9 / 16.2 (68 MB, 4.2 TB/s), 1999 tokens, 32 + 8 + 8 of 128 with mixed
// values 34.8 / 24.9 (98 MB).  A wave's rows that are none are left out: two queries of 64, normed, of 28972 tokens 30.4 -> 20.5,
// 8 + 2 + 2 slots of 64 of 7653 16.3 -> 14.8.  The sums and roundings are those of that kernel (quads_square, two_products): in the order that quads would take by themselves
// 15.6 / 22.4, and the cached rows of a prompt were others.
constexpr int PREP_QUADS = 4;
constexpr int prep_rows(int D) { return PREP_QUADS * 256 / D; }      // rows a wave takes
typedef float quad_u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f32x4 ldq(const float* p) { return *reinterpret_cast<const quad_u*>(p); }
// 1 / root mean square of a row that D / 4 neighbouring lanes hold
template <int D> __device__ __forceinline__ float quad_row_scale(f32x4 x, float eps) { return 1.f / sqrtf(quads_square<D, true>(x) / (float)D + eps); }
template <typename P, int D, int E>
__global__ __launch_bounds__(256) void attn_prep_quads_kernel(float* __restrict__ q, UmbPagedKV kv, const float* __restrict__ proj, int ld,
                                                              const typename El<P>::type* __restrict__ w_q, const typename El<P>::type* __restrict__ w_k,
                                                              const int* __restrict__ pos, const int* __restrict__ slot, const float* __restrict__ freq, int T,
                                                              AttnPrep a, int qk_waves, int waves) {
  typedef typename El<P>::type El_;
  const int item = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6))), lane = threadIdx.x & 63;
  const int t = item / waves, part = item - t * waves;
  if (t >= T) return;
  const int p = pos[t], sl = a.GV ? slot[t] : 0;
  const float* src = proj + (long)t * ld;
  if (part >= qk_waves) {                                    // values
    constexpr int ROWS = prep_rows(E);
    const int sub = lane / (E / 4), e = lane % (E / 4) * 4, first = (part - qk_waves) * ROWS, n = min(ROWS, a.GV - first);
    const float* vs = src + (a.HQ + a.GK) * D;
    const long row0 = ((long)t * a.G + first) * E + e, out0 = a.GV ? pkv_tok(kv, sl, p, first, a.G, E) + e : 0;
    f32x4 v[PREP_QUADS], m[PREP_QUADS];
#pragma unroll
    for (int u = 0; u < PREP_QUADS; ++u) {
      const int r = min(u * (256 / E) + sub, n - 1);
      v[u] = ldq(vs + (first + r) * E + e);
    }
    const float* ms = a.mix.first ? a.mix.first + row0 : vs + first * E + e;      // (no branch between loads: one waits for all of them)
#pragma unroll
    for (int u = 0; u < PREP_QUADS; ++u) m[u] = ldq(ms + min(u * (256 / E) + sub, n - 1) * E);
#pragma unroll
    for (int u = 0; u < PREP_QUADS; ++u) {
      if (u * (256 / E) >= n) break;
      const int r = u * (256 / E) + sub;
      if (a.norm_v) v[u] = v[u] * quad_row_scale<E>(v[u], a.eps);
      if (r >= n) continue;
      if (a.mix.keep) *reinterpret_cast<quad_u*>(a.mix.keep + row0 + r * E) = v[u];
      if (a.mix.first) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[u][i] = fmaf(1.f - a.mix.lambda, v[u][i], a.mix.lambda * m[u][i]);
      }
      st4<P>(reinterpret_cast<El_*>(kv.v) + out0 + (long)r * kv.page * E, v[u]);
    }
    return;
  }
  constexpr int ROWS = prep_rows(D);
  const int sub = lane / (D / 4), e = lane % (D / 4) * 4, first = part * ROWS, n = min(ROWS, a.HQ + a.GK - first), half = a.rot_dims >> 1;
  const bool rot = e < a.rot_dims, low = e < half;
  const int other = a.layout == 0 && rot ? (low ? e + half : e - half) : e;
  const bool far = a.layout == 0 && a.rot_dims > 0;          // partners in another lane's quad
  f32x4 x[PREP_QUADS], y[PREP_QUADS];
#pragma unroll
  for (int u = 0; u < PREP_QUADS; ++u) {
    const float* row = src + (first + min(u * (256 / D) + sub, n - 1)) * D;
    x[u] = ldq(row + e);
    y[u] = ldq(row + other);                                 // (itself where it is in this lane: no branch between loads, one waits for all of them)
  }
  f32x4 cs = {1.f, 1.f, 1.f, 1.f}, sn = {0.f, 0.f, 0.f, 0.f};
  if (rot) {
    // a quad's four angles, or two where it holds whole pairs: one place for the sines, the values go round
    typedef float two __attribute__((ext_vector_type(2), aligned(4)));
    const int at = a.layout == 0 ? (low ? e : e - half) : e >> 1;
    const two f0 = *reinterpret_cast<const two*>(freq + at), f1 = *reinterpret_cast<const two*>(freq + (a.layout == 0 ? at + 2 : at));
    f32x4 fr = {f0[0], f0[1], f1[0], f1[1]};
#pragma unroll 1
    for (int i = a.layout == 0 ? 4 : 2; i > 0; --i) {
      float s, c;
      sincosf((float)p * fr[0], &s, &c);
      fr = f32x4{fr[1], fr[2], fr[3], fr[0]};
      cs = f32x4{cs[1], cs[2], cs[3], c * a.rot_mult};
      sn = f32x4{sn[1], sn[2], sn[3], s * a.rot_mult};
    }
    // x cos - y sin in a pair's first, y cos + x sin in its second
    if (a.layout == 1) {
      cs = f32x4{cs[2], cs[2], cs[3], cs[3]};
      sn = f32x4{-sn[2], sn[2], -sn[3], sn[3]};
    } else if (low) sn = -sn;
  }
  const float temp = attn_temp(a, p);
  const long k0 = a.GK ? pkv_tok(kv, sl, p, 0, a.G, a.maps * D) : 0, k_group = (long)kv.page * a.maps * D;
#pragma unroll
  for (int u = 0; u < PREP_QUADS; ++u) {
    if (u * (256 / D) >= n) break;
    const int r = u * (256 / D) + sub, hs = first + min(r, n - 1), ks = hs - a.HQ;
    const bool is_q = ks < 0;
    if (a.norm_qk) {
      const float f = quad_row_scale<D>(x[u], a.eps);
      x[u] = x[u] * f;
      if (far) y[u] = y[u] * f;
    }
    const El_* w = is_q ? w_q : w_k;
    if (w) {
      x[u] = x[u] * ld4<P>(w + e);
      if (far) y[u] = y[u] * ld4<P>(w + other);
    }
    if (!far) y[u] = f32x4{x[u][1], x[u][0], x[u][3], x[u][2]};
    f32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = two_products(x[u][i], cs[i], y[u][i], sn[i]);
    if (!rot) o = x[u];
    if (r >= n) continue;
    if (is_q) *reinterpret_cast<f32x4*>(q + ((long)t * a.HQ + hs) * D + e) = o * temp;
    else st4<P>(reinterpret_cast<El_*>(kv.k) + k0 + ks / a.maps * k_group + ks % a.maps * D + e, o);
  }
}
// Where it can: whole quads on either side of a pair's distance; weights, queries and cached rows that quads are aligned in.  And where it pays: from five
// slots a token on, of 64 from four, without values from two.  Fewer are one wave of four slots, but two of quads, mostly empty (us, slots four by four / quads,
// bf16, normed, turned, slots of 128: two queries, a key and a value of 67474 tokens 84.5 / 99.3, a query, a key and a value of 85519 112 / 131; three queries, a key
// and a value of 41399 83.6 / 64.6; two queries, a key and a value of 64 of 47362 56.7 / 53.0; two queries of 64 of 28972 23.4 / 20.5).
static inline bool prep_in_quads(const float* q, const UmbPagedKV* kv, const void* w_q, const void* w_k, const AttnPrep& a, int eb) {
  return a.HQ + a.GK + a.GV >= (!a.GV ? 2 : a.D == 64 ? 4 : 5) && (a.D == 64 || a.D == 128) && (a.E == 64 || a.E == 128) && a.rot_dims % (a.layout == 0 ? 8 : 4) == 0 && (uintptr_t)q % 16 == 0 &&
         ((uintptr_t)w_q | (uintptr_t)w_k) % (4 * eb) == 0 && (!a.GV || ((uintptr_t)kv->k | (uintptr_t)kv->v) % (4 * eb) == 0);
}

// The same for many items (rows of at most 128): a wave takes four neighbouring slots of one token, the loads of all four in flight, and
// works the angles out once for them.  A wave per slot was latency times rounds of waves and four times the sines: 1999 tokens of 32 + 16
// slots of 128 42.5 -> 35.0 us (90 MB, 2.6 TB/s); 2300 tokens, 32 + 16 of 64 34 -> 29.
template <typename P>
__global__ __launch_bounds__(256) void attn_prep_four_kernel(float* __restrict__ q, UmbPagedKV kv, const float* __restrict__ proj, int ld,
                                                             const typename El<P>::type* __restrict__ w_q,
                                                             const typename El<P>::type* __restrict__ w_k, const int* __restrict__ pos,
                                                             const int* __restrict__ slot, const float* __restrict__ freq, int T,
                                                             AttnPrep a, int groups) {
  typedef typename El<P>::type El_;
  const int item = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6))), lane = threadIdx.x & 63;
  const int t = item / groups, s0 = item % groups * 4, per = a.HQ + a.GK + a.GV, D = a.D, half = a.rot_dims >> 1;
  if (t >= T) return;
  const int p = pos[t], sl = slot[t];
  int other[2];
  bool rot[2], first[2];
  float x[4][2], y[4][2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int i = lane + 64 * c;
    rot[c] = i < a.rot_dims;
    if (a.layout == 0) { first[c] = i < half; other[c] = first[c] ? i + half : i - half; }
    else { first[c] = (i & 1) == 0; other[c] = i ^ 1; }
    if (!rot[c]) other[c] = 0;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int hs = min(s0 + u, per - 1);
    const bool is_v = hs >= a.HQ + a.GK;
    const int n = is_v ? a.E : D;
    const float* src = proj + (long)t * ld + (is_v ? (a.HQ + a.GK) * D + (hs - a.HQ - a.GK) * a.E : hs * D);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      x[u][c] = lane + 64 * c < n ? src[lane + 64 * c] : 0.f;
      y[u][c] = rot[c] && !is_v ? src[other[c]] : 0.f;
    }
  }
  float cs[2] = {1.f, 1.f}, sn[2] = {0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (rot[c] && s0 < a.HQ + a.GK) {
      const int i = lane + 64 * c;
      sincosf((float)p * freq[a.layout == 0 ? (first[c] ? i : i - half) : i >> 1], &sn[c], &cs[c]);
      sn[c] *= a.rot_mult;
      cs[c] *= a.rot_mult;
    }
  const float temp = a.temp_every > 0 ? 1.f + a.temp_coef * logf((float)((p + 1) / a.temp_every + 1)) : 1.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int hs = s0 + u;
    if (hs >= per) return;
    const bool is_v = hs >= a.HQ + a.GK, is_q = hs < a.HQ;
    const int n = is_v ? a.E : D;
    float f = 1.f;
    if (is_v ? a.norm_v : a.norm_qk) f = 1.f / sqrtf(wave_sum(x[u][0] * x[u][0] + x[u][1] * x[u][1]) / (float)n + a.eps);
    if (is_v) {
      const int g = hs - a.HQ - a.GK;
      El_* row = reinterpret_cast<El_*>(kv.v) + pkv_tok(kv, sl, p, g, a.G, a.E);
      const long o = ((long)t * a.G + g) * a.E;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int i = lane + 64 * c;
        if (i >= n) continue;
        float v = x[u][c] * f;
        if (a.mix.keep) a.mix.keep[o + i] = v;
        if (a.mix.first) v = (1.f - a.mix.lambda) * v + a.mix.lambda * a.mix.first[o + i];
        stf<P>(row + i, v);
      }
      continue;
    }
    const El_* w = is_q ? w_q : w_k;
    const int ks = hs - a.HQ;
    El_* krow = is_q ? nullptr : reinterpret_cast<El_*>(kv.k) + pkv_tok(kv, sl, p, ks / a.maps, a.G, a.maps * D) + (ks % a.maps) * D;
    float* qrow = q + ((long)t * a.HQ + (is_q ? hs : 0)) * D;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int i = lane + 64 * c;
      if (i >= n) continue;
      float v = x[u][c] * f * (w ? ldf<P>(w + i) : 1.f);
      if (rot[c]) {
        const float z = y[u][c] * f * (w ? ldf<P>(w + other[c]) : 1.f);
        v = first[c] ? v * cs[c] - z * sn[c] : v * cs[c] + z * sn[c];
      }
      if (is_q) qrow[i] = v * temp;
      else stf<P>(krow + i, v);
    }
  }
}

constexpr int BSA_MAXC = 8;      // value columns per lane: E <= 512

// positions a token sees: 0 .. kept - 1, then j_lo .. its own; n in all
struct AttnKeys { int j_lo, kept, n; };
__device__ __forceinline__ AttnKeys attn_keys(int i, int window, const UmbAttnForm& form) {
  int j_lo = i - window + 1 > 0 ? i - window + 1 : 0;
  if (form.chunk > 0) j_lo = max(j_lo, i / form.chunk * form.chunk);
  const int kept = min(form.keep_first, j_lo);          // first positions in front of the walk
  return AttnKeys{j_lo, kept, kept + i - j_lo + 1};
}

// a head's sink: fp32, or a latent layer's in storage format
template <typename P, bool LAT> __device__ __forceinline__ float sink_of(const float* sink, int h) {
  if constexpr (LAT) return P::to_f(reinterpret_cast<const u16*>(sink)[h]);
  else return sink[h];
}
// end of a workgroup: the partial sums o_s [nact][RH][Ep], maxima and denominators ml_s [nact][RH][2] (and 2 RH floats behind the nw-th)
// of its waves, added in wave order; nact <= 16: a row's factors are worked out once, by 16 lanes.
// part: this split's result goes there instead ([token][row][split][E + 2] = o .., maximum, denominator)
template <typename P, int RH, int NC, int MAPS, bool LAT = false>
__device__ __forceinline__ void attn_finish(typename El<P>::type* __restrict__ out, int ldo, const float* o_s, int Ep, float* ml_s,
                                            int nact, int nw, float* __restrict__ part, int split, int nsplit,
                                            const float* __restrict__ proj, int ld, int gate_col, int t, int h0, int H, int E,
                                            float out_scale, const UmbAttnForm& form) {
  constexpr int RR = RH / MAPS;
  const int lane = threadIdx.x & 63;
  float* row_s = ml_s + nw * RH * 2;                       // [RH][2] maximum, denominator
  if (threadIdx.x < RH * 16) {
    const int r = threadIdx.x >> 4, w = threadIdx.x & 15;
    float* ml = ml_s + (w * RH + r) * 2;
    const float m = w < nact ? ml[0] : -INFINITY, l = w < nact ? ml[1] : 0.f;
    const float M = row_max16(m), f = m == -INFINITY ? 0.f : expf(m - M), L = row_add16(l * f);
    if (w < nact) ml[0] = f;
    if (w == 0) { row_s[2 * r] = M; row_s[2 * r + 1] = L; }
  }
  __syncthreads();
  auto merged = [&](int r, int d) -> float {               // unnormalised output of row r, column d
    float o = 0.f;
    for (int w = 0; w < nact; ++w) o += o_s[(w * RH + r) * Ep + d] * ml_s[(w * RH + r) * 2];
    return o;
  };
  auto denominator = [&](int r) -> float { return row_s[2 * r + 1] + (form.sink ? expf(sink_of<P, LAT>(form.sink, h0 + r / MAPS) - row_s[2 * r]) : 0.f); };
  auto gate_of = [&](int h, int d) {
    return gate_col >= 0 ? 1.f / (1.f + expf(-proj[(long)t * ld + gate_col + (form.gate_elem ? h * E + d : h)])) : 1.f;
  };
  if ((MAPS == 1 || part) && E % 4 == 0 && Ep % 4 == 0) {  // four columns a thread: a column a thread was up to eight rounds of the waves' sums
    typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
    const int per = E >> 2;
    for (int x = threadIdx.x; x < RH * per; x += nw * 64) {
      const int r = x / per, d = x % per * 4;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
      for (int w = 0; w < nact; ++w) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(o_s + (w * RH + r) * Ep + d);
        const float f = ml_s[(w * RH + r) * 2];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += v[e] * f;
      }
      if (part) {
        float* pr = part + ((((long)t * H + h0) * MAPS + r) * nsplit + split) * (E + 2);
        *reinterpret_cast<quad*>(pr + d) = o;
        if (d == 0) { pr[E] = row_s[2 * r]; pr[E + 1] = row_s[2 * r + 1]; }
        continue;
      }
      const float L = denominator(r);
#pragma unroll
      for (int e = 0; e < 4; ++e) stf<P>(out + (long)t * ldo + (long)(h0 + r) * E + d + e, out_scale * gate_of(h0 + r, d + e) * (o[e] / L));
    }
  } else if (MAPS == 1 || part) {
    for (int x = threadIdx.x; x < RH * E; x += nw * 64) {
      const int r = x / E, d = x % E;
      const float o = merged(r, d);
      if (part) {
        float* pr = part + ((((long)t * H + h0) * MAPS + r) * nsplit + split) * (E + 2);
        pr[d] = o;
        if (d == 0) { pr[E] = row_s[2 * r]; pr[E + 1] = row_s[2 * r + 1]; }
        continue;
      }
      stf<P>(out + (long)t * ldo + (long)(h0 + r) * E + d, out_scale * gate_of(h0 + r, d) * (o / denominator(r)));
    }
  } else {
    // a wave per head: o = a1 - lambda a2 over its root mean square
    for (int rr = threadIdx.x >> 6; rr < RR; rr += nw) {
      float v[NC], u[NC], ss = 0.f;
      const float L1 = denominator(MAPS * rr), L2 = denominator(MAPS * rr + MAPS - 1);
#pragma unroll
      for (int c = 0; c < NC; ++c) v[c] = u[c] = 0.f;
#pragma unroll 1
      for (int w = 0; w < nact; ++w) {                       // all columns of both maps side by side
        const int r1 = w * RH + MAPS * rr, r2 = r1 + MAPS - 1;
        const float f1 = ml_s[r1 * 2], f2 = ml_s[r2 * 2];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int d = min(lane + 64 * c, E - 1);
          v[c] += o_s[r1 * Ep + d] * f1;
          u[c] += o_s[r2 * Ep + d] * f2;
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const float o = v[c] / L1 - form.lambda * (u[c] / L2);
        v[c] = o;
        if (lane + 64 * c < E) ss += o * o;
      }
      ss = wave_sum(ss);
      const float f = out_scale / sqrtf(ss / (float)E + form.eps);
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (lane + 64 * c < E) stf<P>(out + (long)t * ldo + (long)(h0 + rr) * E + lane + 64 * c, v[c] * f * gate_of(h0 + rr, lane + 64 * c));
    }
  }
}

// RH rows of the workgroup = RH / MAPS query heads with MAPS maps each (row r: head r / MAPS, map r % MAPS)
template <typename P, int RH, int NC, int NW, int MAPS>
__global__ __launch_bounds__(NW * 64) void bsa_attend_kernel(typename El<P>::type* __restrict__ out, int ldo,
                                                             const float* __restrict__ q, UmbPagedKV kv,
                                                             const float* __restrict__ proj, int ld, int gate_col,
                                                             const float* __restrict__ bias, int n_dist,
                                                             const int* __restrict__ pos, const int* __restrict__ slot_, int H,
                                                             int G, int D, int E, int window, float scale, float out_scale,
                                                             float softcap, UmbAttnForm form, float* __restrict__ part,
                                                             int nsplit) {
  static_assert(RH % MAPS == 0, "rows are whole heads");
  typedef typename El<P>::type El_;
  extern __shared__ float lds[];
  constexpr int KB = 8;
  const int split = blockIdx.z;                         // nsplit > 1: the workgroup takes every nsplit-th group of NW rounds
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int Dp = (D + 3) & ~3, Ep = (E + 3) & ~3, Mp = Dp > Ep ? Dp : Ep;
  // [RH][Dp] queries (later [NW][RH][Ep] partial sums), [NW][2 RH] maxima and denominators, per wave [RH][64] weights + offsets
  float* q_s = lds;
  float* ml_s = lds + NW * RH * Mp;
  float* w_s = ml_s + NW * 2 * RH + wave * (RH * 64 + 128);
  long* off_s = reinterpret_cast<long*>(w_s + RH * 64);
  const int t = blockIdx.x, hpg = H / G;
  constexpr int RR = RH / MAPS;
  const int h0 = blockIdx.y * RR, g = h0 / hpg;           // RR divides H / G: the block's heads share key/value head g
  const int i = pos[t], slot = slot_[t];
  for (int x = threadIdx.x; x < RH * D; x += NW * 64) {
    const int r = x / D, d = x % D;
    q_s[r * Dp + d] = q[(((long)t * H + h0) * MAPS + r) * D + d];
  }
  __syncthreads();
  const AttnKeys keys = attn_keys(i, window, form);
  const int j_lo = keys.j_lo, kept = keys.kept, n_keys = keys.n;
  const bool vec = (D & 7) == 0 && sizeof(El_) == 2;
  float acc[RH][NC], m_run[RH], l_run[RH];
#pragma unroll
  for (int r = 0; r < RH; ++r) {
    m_run[r] = -INFINITY;
    l_run[r] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[r][c] = 0.f;
  }
  int dcl[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) dcl[c] = lane + 64 * c < E ? lane + 64 * c : E - 1;
  for (int base = (split * NW + wave) * 64; base < n_keys; base += nsplit * NW * 64) {
    const int kx = base + lane;
    float s[RH];
#pragma unroll
    for (int r = 0; r < RH; ++r) s[r] = 0.f;
    long off = 0;
    int dist = 0;
    if (kx < n_keys) {
      const int j = kx < kept ? kx : j_lo + kx - kept;
      dist = i - j;
      const El_* kr = reinterpret_cast<const El_*>(kv.k) + pkv_tok(kv, slot, j, g, G, MAPS * D);
      off = pkv_tok(kv, slot, j, g, G, E);
      bool done = false;
      if constexpr (sizeof(El_) == 2) {
        if (vec) {
#pragma unroll
          for (int mp = 0; mp < MAPS; ++mp)
          for (int d = 0; d < D; d += 64) {              // eight 16-byte loads in flight, then their 64 x RH products
            u32x4 kk[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) kk[u] = *reinterpret_cast<const u32x4*>(kr + mp * D + (d + 8 * u < D ? d + 8 * u : 0));
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              if (d + 8 * u >= D) break;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float k0 = lo_f<P>(kk[u][e]), k1 = hi_f<P>(kk[u][e]);
                const int dd = d + 8 * u + 2 * e;
#pragma unroll
                for (int r = mp; r < RH; r += MAPS) s[r] += q_s[r * Dp + dd] * k0 + q_s[r * Dp + dd + 1] * k1;
              }
            }
          }
          done = true;
        }
      }
      if (!done) {
#pragma unroll
        for (int mp = 0; mp < MAPS; ++mp)
          for (int d = 0; d < D; ++d) {
            const float kd = ldf<P>(kr + mp * D + d);
#pragma unroll
            for (int r = mp; r < RH; r += MAPS) s[r] += q_s[r * Dp + d] * kd;
          }
      }
    }
    const int bi = dist < n_dist ? dist : n_dist - 1;
#pragma unroll
    for (int r = 0; r < RH; ++r) {
      float sc = s[r] * scale;
      if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);          // capped score; the bias (if any) is added to the capped value
      const float sv = kx < n_keys ? sc + (bias ? bias[(long)(h0 + r / MAPS) * n_dist + bi] : 0.f) : -INFINITY;
      const float m_new = fmaxf(m_run[r], wave_max(sv));          // finite: every round has at least one key
      const float fac = expf(m_run[r] - m_new);                   // 0 on the first round (m_run = -inf)
      const float pw = kx < n_keys ? expf(sv - m_new) : 0.f;
      l_run[r] = l_run[r] * fac + wave_sum(pw);
      m_run[r] = m_new;
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[r][c] *= fac;
      w_s[r * 64 + lane] = pw;
    }
    off_s[lane] = off;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int cnt = n_keys - base < 64 ? n_keys - base : 64;
    for (int j0 = 0; j0 < cnt; j0 += KB) {
      float vv[KB][NC];
#pragma unroll
      for (int u = 0; u < KB; ++u) {
        const long oj = off_s[j0 + u < cnt ? j0 + u : cnt - 1];
#pragma unroll
        for (int c = 0; c < NC; ++c) vv[u][c] = ldf<P>(reinterpret_cast<const El_*>(kv.v) + oj + dcl[c]);
      }
#pragma unroll
      for (int u = 0; u < KB; ++u) {
#pragma unroll
        for (int r = 0; r < RH; ++r) {
          const float wj = j0 + u < cnt ? w_s[r * 64 + j0 + u] : 0.f;
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[r][c] += wj * vv[u][c];
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();                                  // every wave is done with the queries: their LDS becomes the partials
#pragma unroll
  for (int r = 0; r < RH; ++r) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = lane + 64 * c;
      if (d < E) lds[(wave * RH + r) * Ep + d] = acc[r][c];
    }
    if (lane == 0) { ml_s[(wave * RH + r) * 2] = m_run[r]; ml_s[(wave * RH + r) * 2 + 1] = l_run[r]; }
  }
  __syncthreads();
  attn_finish<P, RH, NC, MAPS>(out, ldo, lds, Ep, ml_s, NW, NW, nsplit > 1 ? part : nullptr, split, nsplit, proj, ld, gate_col, t, h0, H, E,
                               out_scale, form);
}

// Attention of single tokens (see seq_decode.h).  Workgroup = (token, RH rows of one key/value head, split); its waves deal the rounds of
// 16 keys among themselves.  With nsplit > 1 workgroup z takes the spans of ATT_SPAN keys z, z + nsplit, ..; a token whose keys fit one
// span is finished by workgroup 0 and the others leave at once, so a short context pays neither the split nor the merge.
// Before -> now, replayed from a graph: 48 tokens behind 40 keys of 64 features 19.1 -> 6.2 us, behind 500 29.4 -> 20.5; one token behind
// 40 / 2000 keys of 128 features 16.0 -> 7.4 / 19.2 -> 12.8 (spans of 1024: 22.0); two maps, values of 256, one token behind 40 / 1000
// 23.0 -> 9.5 / 27.2 -> 19.8; 64 tokens behind 1000, 128 features, 81 -> 51 (262 MB of rows, 5.1 TB/s).
// Few rows in all go two to a workgroup and not four: a wave's products halve and twice the units have some (one token, two maps of 128 | 256 behind 77 keys 9.7 -> 8.7 us,
// a sink of 128 7.4 -> 6.3, 32 + 8 heads of 128 behind 2000 12.4 -> 10.2).
// LAT: latent attention (one row a token for all heads, kv.k; its first E columns are the values).  A round of 16 keys of it is some 4 us of one wave's products,
// so a span that goes to a workgroup of its own is 64 keys, four waves.  us, rounds of 64 keys with a key a lane and single columns a lane (lat_attend_kernel, which
// keeps the other shapes) / this with the merge, 32 heads of 512 + 64: one token behind 40 / 300 / 2000 keys (1024 of a window) 23.3 / 30.9 / 57.6 -> 9.9 / 12.1 / 12.8,
// 16 behind 100 29.5 -> 14.4, 40 behind 100 82 -> 27.6; 16 heads of 256 + 32: one behind 40 / 2000 19.7 / 26.0 -> 7.2 / 9.4, 40 behind 60 23.0 -> 8.4.
constexpr int ATT_SPAN = 256, LAT_SPAN = 64;

// PREP: steps of one token a sequence.  The queries come from the projection and the token's key and value with them (attn_prep above, which a launch of
// its own did in 4 - 5 us): the key and value stand in LDS for this workgroup, whose last round takes them from there -- what the cache holds at the token's
// position is not there yet -- and the group's first workgroup appends them.
// A launch is latency, a fifth of it the fetch of code that is executed once: one place for queries and keys, an angle a pair, loops not unrolled where a
// round is enough; and the first round's rows asked for in front of the preparation (us a launch inside a step, 20 / 16 KB of code: one token, two maps of
// 128 | 256 10.3 / 7.9, sink heads of 128 8.0 / 7.1; 48 tokens, heads of 64 10.1 / 9.2).
struct DecodePrep { AttnPrep a; const void *w_q, *w_k; const float* freq; };
// (One map, by four waves, prepared: as many workgroups a unit as an element a lane's preparation left, of which the pairs' registers would cost one -- three for
// values of 256: 400 tokens, heads of 256, 300 keys 112 / 125 us; four for values of 128 in fp16: 32 heads of 64 | 128, 125 tokens of 12 keys 10.3 / 15.7, 99 of 2463
// keys 187 / 234.  In bf16 they are three either way: held to four some values spill, 118 tokens of 11 keys 15.9 -> 10.5, but 150 of 1464 keys 167 -> 199.)
template <typename P> constexpr int decode_waves(int LPR, int NW, int MAPS, bool PREP) {
  return !PREP || MAPS > 1 || NW != 4 ? 1 : LPR == 32 ? 3 : LPR == 16 && std::is_same<P, F16>::value ? 4 : 1;
}
template <typename P, int RH, int LPR, int NW, int MAPS, bool LAT = false, bool PREP = false>
__global__ __launch_bounds__(NW * 64, decode_waves<P>(LPR, NW, MAPS, PREP))
void attn_decode_kernel(u16* __restrict__ out, int ldo, const float* __restrict__ q, UmbPagedKV kv,
                                                              const float* __restrict__ proj, int ld, int gate_col,
                                                              const float* __restrict__ bias, int n_dist, const int* __restrict__ pos,
                                                              const int* __restrict__ slot_, int H, int G, int D, int window, float scale,
                                                              float out_scale, float softcap, UmbAttnForm form, float* __restrict__ part,
                                                              int nsplit, DecodePrep prep) {
  constexpr int E = LPR * 8, KPI = 64 / LPR, VL = 16 / KPI, RR = RH / MAPS;
  constexpr int SPAN = LAT ? LAT_SPAN : ATT_SPAN;
  static_assert(!LAT || MAPS == 1, "one map");
  const int ldv = LAT ? D : E;                             // elements between two value rows
  extern __shared__ float lds[];
  const int split = blockIdx.z, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 15, quarter = lane >> 4;
  float* q_s = lds;                                        // [RH][D]
  u16* new_k = reinterpret_cast<u16*>(lds + RH * D);       // [MAPS][D], the token's own, and its value [E]
  u16* new_v = new_k + MAPS * D;
  float* o_s = lds + RH * D + (PREP ? (MAPS * D + E) / 2 : 0);               // [NW][RH][E]
  float* ml_s = o_s + NW * RH * E;                         // [NW][RH][2], [RH][2]
  const int t = blockIdx.x, h0 = blockIdx.y * RR, g = h0 / (H / G);
  const int i = pos[t], slot = slot_[t];
  const AttnKeys keys = attn_keys(i, window, form);
  const int first = split * SPAN;
  if (first >= keys.n) return;
  const int nact = min(NW, ((nsplit > 1 ? min(keys.n - first, SPAN) : keys.n) + 15) / 16);       // waves that get a round
  auto key_pos = [&](int kx) { return kx < keys.kept ? kx : keys.j_lo + kx - keys.kept; };
  int base = first + wave * 16;
  unsigned row = 0;
  if (wave < nact) row = pkv_tok_row(kv, slot, key_pos(min(base + j, keys.n - 1)), g, G);
  typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
  // The first round's rows are on their way while the token's own are prepared, which is as long as their trip: a lane asks for one word of each, its
  // quarter's (all lines of a row up to 512 bytes), and the round finds them near.  Held in registers instead they cost the kernel of four rows a wave a SIMD.
  // Only where a wave has one round: of more the first is a small part, and asking twice took longer than it gave (two maps of 64, 2000 keys of two tokens
  // 25.4 / 27.6 us).
  const bool early = PREP && keys.n <= NW * 16;
  unsigned near_k = 0, near_v = 0;
  float bv[RR];
  auto biases = [&]() {
    const int dist = i - key_pos(min(base + j, keys.n - 1)), bi = dist < n_dist ? dist : n_dist - 1;
#pragma unroll
    for (int r = 0; r < RR; ++r) bv[r] = bias ? bias[(long)(h0 + r) * n_dist + bi] : 0.f;
  };
  if (wave < nact) {
    if (early) near_k = *reinterpret_cast<const unsigned*>(reinterpret_cast<const u16*>(kv.k) + (long)row * (MAPS * D) + quarter * (MAPS * D / 4));
    if (early && !LAT) near_v = *reinterpret_cast<const unsigned*>(reinterpret_cast<const u16*>(kv.v) + (long)row * E + quarter * (E / 4));
    if (PREP) biases();
  }
  if constexpr (PREP) {
    const AttnPrep& a = prep.a;
    const float* src = proj + (long)t * ld;
    const bool append = split == 0 && h0 % (H / G) == 0;
    const float temp = attn_temp(a, i);
#pragma unroll 1
    for (int task = wave; task < RH + (a.GK ? MAPS + 1 : 0); task += NW) {       // a row a wave
      if (task < RH + MAPS) {
        const bool is_q = task < RH;
        const int mp = task - RH;
        u16* row_k = is_q ? nullptr : reinterpret_cast<u16*>(kv.k) + pkv_tok(kv, slot, i, g, G, MAPS * D) + mp * D;
        attn_prep_pairs<P>(src + (is_q ? h0 * MAPS + task : a.HQ + g * MAPS + mp) * D, a, reinterpret_cast<const u16*>(is_q ? prep.w_q : prep.w_k), prep.freq, i,
                           is_q ? temp : 1.f, [&](int x, float v) {
          if (is_q) {
            q_s[task * D + x] = v;
            return;
          }
          const u16 b = P::from_f(v);
          new_k[mp * D + x] = b;
          if (append) row_k[x] = b;
        });
      } else {
        u16* row_v = reinterpret_cast<u16*>(kv.v) + pkv_tok(kv, slot, i, g, G, E);
        attn_prep_value_few<(E + 63) / 64>(src + (a.HQ + a.GK) * D + g * E, a, ((long)t * G + g) * E, append, [&](int x, float v) {
          const u16 b = P::from_f(v);
          new_v[x] = b;
          if (append) row_v[x] = b;
        });
      }
    }
  } else {
    for (int x = threadIdx.x; x < RH * D / 4; x += NW * 64)      // (D: a multiple of 32)
      *reinterpret_cast<f32x4*>(q_s + 4 * x) = *reinterpret_cast<const quad*>(q + ((long)t * H + h0) * MAPS * D + 4 * x);
  }
  __syncthreads();
  if (wave < nact) {
    if (PREP) asm volatile("" :: "v"(near_k), "v"(near_v));  // (asked for, whatever they hold; no registers in the rounds)
    float acc[RH * 8], m_run[RH], l_run[RH];
#pragma unroll
    for (int r = 0; r < RH; ++r) { m_run[r] = -INFINITY; l_run[r] = 0.f; }
#pragma unroll
    for (int v = 0; v < RH * 8; ++v) acc[v] = 0.f;
    const u16* vcol = reinterpret_cast<const u16*>(LAT ? kv.k : kv.v) + (lane & (LPR - 1)) * 8;
    while (base < keys.n) {
      const int kx = base + j;
      u32x4 vv[VL];
#pragma unroll
      for (int u = 0; u < VL; ++u) vv[u] = *reinterpret_cast<const u32x4*>(vcol + (long)(unsigned)__shfl((int)row, KPI * u + lane / LPR, 64) * ldv);
      // the round with the token's own key: it and the lanes behind the last key (whose weights are 0) take what LDS has
      const bool own = PREP && prep.a.GK && base + 16 >= keys.n;
      if (own) {
#pragma unroll
        for (int u = 0; u < VL; ++u)
          if (base + KPI * u + lane / LPR >= keys.n - 1) vv[u] = *reinterpret_cast<const u32x4*>(new_v + (lane & (LPR - 1)) * 8);
      }
      const u16* kr = reinterpret_cast<const u16*>(kv.k) + (long)row * (MAPS * D) + quarter * 8;
      if (!PREP) biases();                                   // (a round ahead, two maps of 128 | 256, 400 tokens of 16 keys: 38.5 -> 46.7 us)
      // the next round of this wave: NW rounds on, or in the next of its workgroup's spans
      int next = base + NW * 16;
      if (nsplit > 1 && next / SPAN != base / SPAN) next += (nsplit - 1) * SPAN;
      unsigned next_row = 0;
      if (next < keys.n) next_row = pkv_tok_row(kv, slot, key_pos(min(next + j, keys.n - 1)), g, G);
      float s[RH];
#pragma unroll
      for (int r = 0; r < RH; ++r) s[r] = 0.f;
#pragma unroll 1
      for (int d = 0; d < D; d += 128) {
        u32x4 kk[MAPS][4];
#pragma unroll
        for (int mp = 0; mp < MAPS; ++mp)
#pragma unroll
          for (int u = 0; u < 4; ++u) kk[mp][u] = *reinterpret_cast<const u32x4*>(kr + mp * D + (d + 32 * u < D ? d + 32 * u : 0));
        if (own) {
#pragma unroll
          for (int mp = 0; mp < MAPS; ++mp)
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (kx >= keys.n - 1) kk[mp][u] = *reinterpret_cast<const u32x4*>(new_k + mp * D + (d + 32 * u < D ? d + 32 * u : 0) + quarter * 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (d + 32 * u >= D) break;
#pragma unroll
          for (int mp = 0; mp < MAPS; ++mp) {
            float kf[8];
            unpack8<P>(kk[mp][u], kf);
#pragma unroll
            for (int r = mp; r < RH; r += MAPS) {
              const f32x4 qa = *reinterpret_cast<const f32x4*>(q_s + r * D + d + 32 * u + quarter * 8);
              const f32x4 qb = *reinterpret_cast<const f32x4*>(q_s + r * D + d + 32 * u + quarter * 8 + 4);
#pragma unroll
              for (int e = 0; e < 4; ++e) s[r] += qa[e] * kf[e];
#pragma unroll
              for (int e = 0; e < 4; ++e) s[r] += qb[e] * kf[4 + e];
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < RH; ++r) s[r] = add_rows(s[r]) * scale;
      if (softcap > 0.f) {
#pragma unroll
        for (int r = 0; r < RH; ++r) s[r] = softcap * tanhf(s[r] / softcap);
      }
#pragma unroll
      for (int r = 0; r < RH; ++r) {
        const float sv = kx < keys.n ? s[r] + bv[r / MAPS] : -INFINITY;
        const float m_new = fmaxf(m_run[r], row_max16(sv));
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;          // a round of -inf scores alone: weights 0, nothing to rescale
        const float fac = expf(m_run[r] - m_ref);
        s[r] = kx < keys.n ? expf(sv - m_ref) : 0.f;
        l_run[r] = l_run[r] * fac + s[r];
        m_run[r] = m_new;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r * 8 + e] *= fac;
      }
#pragma unroll
      for (int u = 0; u < VL; ++u) {
        float vf[8];
        unpack8<P>(vv[u], vf);
#pragma unroll
        for (int r = 0; r < RH; ++r) {
          const float w = __shfl(s[r], KPI * u + lane / LPR, 64);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[r * 8 + e] += w * vf[e];
        }
      }
      base = next;
      row = next_row;
      if (PREP && base < keys.n) biases();
    }
#pragma unroll
    for (int r = 0; r < RH; ++r) {
      const float l = row_add16(l_run[r]);
      if (lane == 0) { ml_s[(wave * RH + r) * 2] = m_run[r]; ml_s[(wave * RH + r) * 2 + 1] = l; }
    }
    store_groups<RH, LPR>(o_s + wave * RH * E, acc, lane);
  }
  __syncthreads();
  attn_finish<P, RH, (E + 63) / 64, MAPS, LAT>(out, ldo, o_s, E, ml_s, nact, NW, keys.n > SPAN && nsplit > 1 ? part : nullptr, split, nsplit,
                                          proj, ld, gate_col, t, h0, H, E, out_scale, form);
}

// the splits of one (token, head) merged: lane s holds split s's maximum and denominator (a split that had no key carries
// M = -inf, L = 0), the factors go round by shuffles, every sum runs over the splits in order
// (one map: a wave for every 64 columns, each with the factors of its own; 64 columns after the other were a round trip each)
template <typename P, int MAPS, bool LAT = false>
__global__ __launch_bounds__(MAPS == 1 ? 512 : 64) void bsa_merge_kernel(typename El<P>::type* __restrict__ out, int ldo, const float* __restrict__ part,
                                                       const float* __restrict__ proj, int ld, int gate_col, int H, int E,
                                                       int splits, float out_scale, UmbAttnForm form, const int* __restrict__ pos,
                                                       int window) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
  int nsplit = splits;
  if (window > 0) {                                       // splits by spans: those that had keys, none if one workgroup did it all
    const int n = attn_keys(pos[t], window, form).n;
    if (n <= (LAT ? LAT_SPAN : ATT_SPAN)) return;
    nsplit = min(splits, (n + (LAT ? LAT_SPAN : ATT_SPAN) - 1) / (LAT ? LAT_SPAN : ATT_SPAN));
  }
  auto gate_of = [&](int d) {
    return gate_col >= 0 ? 1.f / (1.f + expf(-proj[(long)t * ld + gate_col + (form.gate_elem ? h * E + d : h)])) : 1.f;
  };
  const float* pr[MAPS];
  float f[MAPS][16], inv[MAPS];
#pragma unroll
  for (int mp = 0; mp < MAPS; ++mp) {
    pr[mp] = part + (((long)t * H + h) * MAPS + mp) * splits * (E + 2);
    const float ms = lane < nsplit ? pr[mp][lane * (E + 2) + E] : -INFINITY;
    const float ls = lane < nsplit ? pr[mp][lane * (E + 2) + E + 1] : 0.f;
    const float M = wave_max(ms);
    const float fs = ms == -INFINITY ? 0.f : expf(ms - M);
    float L = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      f[mp][s] = __shfl(fs, s, 64);
      L += __shfl(ls * fs, s, 64);
    }
    if (form.sink) L += expf(sink_of<P, LAT>(form.sink, h) - M);
    inv[mp] = 1.f / L;
  }
  auto column = [&](int mp, int d) -> float {
    float v[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) v[s] = pr[mp][(s < nsplit ? s : nsplit - 1) * (E + 2) + d];
    float o = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) o += s < nsplit ? v[s] * f[mp][s] : 0.f;
    return o * inv[mp];
  };
  typename El<P>::type* orow = out + (long)t * ldo + (long)h * E;
  if constexpr (MAPS == 1) {
    for (int d = threadIdx.x; d < E; d += blockDim.x) stf<P>(orow + d, column(0, d) * (out_scale * gate_of(d)));
  } else {
    float v[BSA_MAXC], ss = 0.f;
#pragma unroll
    for (int c = 0; c < BSA_MAXC; ++c) {
      const int d = lane + 64 * c;
      if (64 * c < E) {                                  // uniform
        const float o = d < E ? column(0, d) - form.lambda * column(1, d) : 0.f;
        v[c] = o;
        ss += o * o;
      }
    }
    ss = wave_sum(ss);
    const float c0 = out_scale / sqrtf(ss / (float)E + form.eps);
#pragma unroll
    for (int c = 0; c < BSA_MAXC; ++c)
      if (lane + 64 * c < E) stf<P>(orow + lane + 64 * c, v[c] * (c0 * gate_of(lane + 64 * c)));
  }
}

static inline bool form_ok(const UmbAttnForm* f) { return !f || ((f->maps == 1 || f->maps == 2) && f->chunk >= 0 && f->keep_first >= 0); }
static inline int form_gate_cols(const UmbAttnForm& f, int H, int E) { return f.gate_elem ? H * E : H; }

static inline bool prep_ok(const UmbPagedKV* kv, const float* proj, int ld, int append, const int* pos, const int* slot, const float* freq, int rot_dims,
                           int layout, int T, int H, int G, int D, int E, int maps) {
  return !(T < 1 || H < 1 || G < 1 || H % G || D < 1 || E < 1 || maps < 1 || maps > 2 || rot_dims < 0 || rot_dims > D || (rot_dims & 1) ||
           (rot_dims && !freq) || layout < 0 || layout > 1 || (append && !bsa_kv_ok(kv)) || !proj || !pos || !slot ||
           ld < maps * H * D + (append ? maps * G * D + G * E : 0));
}
static inline AttnPrep prep_of(int append, int norm_qk, int norm_v, int rot_dims, int layout, float rot_mult, int H, int G, int D, int E, int maps,
                               float temp_coef, int temp_every, float eps, const UmbValueMix* mix) {
  return AttnPrep{maps * H, append ? maps * G : 0, G, append ? G : 0, D, E, maps, norm_qk, norm_v, rot_dims, layout, rot_mult,
                  temp_coef, temp_every, eps, mix ? *mix : UmbValueMix{nullptr, nullptr, 0.f, 0.f}};
}
extern "C" int umb_attn_prep_mix(float* q, const UmbPagedKV* kv, const float* proj, int ld, int append, const void* w_q, const void* w_k,
                                 int norm_qk, int norm_v, const int* pos, const int* slot, const float* freq, int rot_dims, int layout,
                                 float rot_mult, int T, int H, int G, int D, int E, int maps, float temp_coef, int temp_every, float eps,
                                 const UmbValueMix* mix, int dtype, hipStream_t st) {
  if (!q || !prep_ok(kv, proj, ld, append, pos, slot, freq, rot_dims, layout, T, H, G, D, E, maps)) return UMB_EINVAL;
  const AttnPrep a = prep_of(append, norm_qk, norm_v, rot_dims, layout, rot_mult, H, G, D, E, maps, temp_coef, temp_every, eps, mix);
  const UmbPagedKV none{};
  const long items = (long)T * (a.HQ + a.GK + a.GV);
  // from three rounds of waves over the chip on (us, a wave each / four: 17600 items of two maps 9.2 / 10.5, 19200 of 64 10.2 / 9.9, 30800 of two maps
  // 13.9 / 13.5, 96000 37.9 / 29.3)
  if (items >= 24576 && prep_in_quads(q, kv, w_q, w_k, a, dtype == UMB_SEQ_F32 ? 4 : 2)) {
    const int qk = (a.HQ + a.GK + prep_rows(D) - 1) / prep_rows(D), waves = qk + (a.GV + prep_rows(E) - 1) / prep_rows(E);
#define QUADS(DD, EE) hipLaunchKernelGGL((attn_prep_quads_kernel<P, DD, EE>), dim3((unsigned)(((long)T * waves + 3) / 4)), dim3(256), 0, st, q, append ? *kv : none, \
                                         proj, ld, (const typename El<P>::type*)w_q, (const typename El<P>::type*)w_k, pos, slot, freq, T, a, qk, waves)
    DISPATCH_SEQ_DTYPE(dtype, {
      if (D == 64 && E == 64) QUADS(64, 64);
      else if (D == 64) QUADS(64, 128);
      else if (E == 64) QUADS(128, 64);
      else QUADS(128, 128);
    })
#undef QUADS
    UMB_LAUNCH_CHECK();
    return UMB_OK;
  }
  if (items >= 24576 && D <= 128 && E <= 128) {
    const int groups = (a.HQ + a.GK + a.GV + 3) / 4;
    DISPATCH_SEQ_DTYPE(dtype, {
      typedef typename El<P>::type El_;
      hipLaunchKernelGGL(attn_prep_four_kernel<P>, dim3((unsigned)(((long)T * groups + 3) / 4)), dim3(256), 0, st, q, append ? *kv : none, proj,
                         ld, (const El_*)w_q, (const El_*)w_k, pos, slot, freq, T, a, groups);
    })
    UMB_LAUNCH_CHECK();
    return UMB_OK;
  }
  DISPATCH_SEQ_DTYPE(dtype, {
    typedef typename El<P>::type El_;
    hipLaunchKernelGGL(attn_prep_kernel<P>, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, st, q, append ? *kv : none, proj, ld,
                       (const El_*)w_q, (const El_*)w_k, pos, slot, freq, T, a);
  })
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_attn_prep(float* q, const UmbPagedKV* kv, const float* proj, int ld, int append, const void* w_q, const void* w_k,
                             int norm_qk, int norm_v, const int* pos, const int* slot, const float* freq, int rot_dims, int layout,
                             float rot_mult, int T, int H, int G, int D, int E, int maps, float temp_coef, int temp_every, float eps,
                             int dtype, hipStream_t st) {
  return umb_attn_prep_mix(q, kv, proj, ld, append, w_q, w_k, norm_qk, norm_v, pos, slot, freq, rot_dims, layout, rot_mult, T, H, G, D, E,
                           maps, temp_coef, temp_every, eps, nullptr, dtype, st);
}

extern "C" int umb_bsa_prep(float* q, const UmbPagedKV* kv, const float* proj, int ld, const void* w_q, const void* w_k,
                            const int* pos, const int* slot, int T, int H, int G, int D, int E, float temp_coef, int temp_every,
                            float eps, int dtype, hipStream_t st) {
  return umb_attn_prep(q, kv, proj, ld, 1, w_q, w_k, 1, 1, pos, slot, nullptr, 0, 0, 1.f, T, H, G, D, E, 1, temp_coef, temp_every, eps,
                       dtype, st);
}

template <typename P, int RH, int NC, int NW, int MAPS>
static int bsa_launch(dim3 grid, size_t lds, hipStream_t st, void* out, int ldo, const float* q, const UmbPagedKV& kv,
                      const float* proj, int ld, int gate_col, const float* bias, int n_dist, const int* pos, const int* slot, int H,
                      int G, int D, int E, int window, float scale, float out_scale, float softcap, const UmbAttnForm& form,
                      float* scratch, int nsplit) {
  typedef typename El<P>::type El_;
  if (ensure_dynamic_lds<bsa_attend_kernel<P, RH, NC, NW, MAPS>>(lds) != UMB_OK) return UMB_EHIP;
  hipLaunchKernelGGL((bsa_attend_kernel<P, RH, NC, NW, MAPS>), grid, dim3(NW * 64), lds, st, (El_*)out, ldo, q, kv, proj, ld, gate_col,
                     bias, n_dist, pos, slot, H, G, D, E, window, scale, out_scale, softcap, form, scratch, nsplit);
  return UMB_OK;
}

// workgroups that one item's spans of keys are dealt to; most: keys a token can have, floats: of one split of all items
static inline int decode_splits(int span, long items, long most, long floats, const float* scratch, long scratch_floats) {
  int nsplit = 1;
  if (scratch && items <= 64 && most > span) {
    nsplit = (int)(512 / items) < 16 ? (int)(512 / items) : 16;
    if (nsplit > (most + span - 1) / span) nsplit = (int)((most + span - 1) / span);
    while (nsplit > 1 && floats * nsplit > scratch_floats) nsplit >>= 1;
  }
  return nsplit;
}
// the decode kernel: spans of ATT_SPAN keys dealt to several workgroups only where few items leave the chip idle; 16 waves per item as
// long as every item gets a compute unit of its own (values of 256: their registers do not hold it), 8 while two share one, 4 beyond
// (us with 8 / 4 waves, 32 + 8 heads of 128: 1024 items behind 30 / 200 keys 12.8 / 8.4, 30.2 / 27.5; 512 items behind 500 28.8 / 36.7)
template <typename P>
static int attn_decode(void* out, int ldo, const float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col, const float* bias,
                       int n_dist, const int* pos, const int* slot, int T, int H, int G, int D, int E, int window, float scale,
                       float out_scale, float softcap, const UmbAttnForm& form, float* scratch, long scratch_floats, hipStream_t st,
                       const DecodePrep* prep = nullptr) {
  const int maps = form.maps, hpg = H / G;
  int rh = (long)T * H * maps <= 128 ? 2 : 4;
  while (rh > maps && hpg % (rh / maps)) rh >>= 1;
  const int hblocks = H * maps / rh;
  const long items = (long)T * hblocks;
  // keys a token can have: by the mask's form and by the pages there are (a page table has room for the whole pool).  So this sees only a pool that is one
  // span of keys altogether, a single short conversation's: nobody splits there, and the merge behind it would find nothing to do (one token of 8B
  // widths in a cache of 192 positions, three layers 56 us -> 41 without the merges, 4.6 us each).  In a larger pool a short sequence's merge still runs.
  const long most = std::min((long)(form.chunk > 0 && form.chunk < window ? form.chunk : window) + form.keep_first, (long)kv->max_pages * kv->page);
  const int nsplit = decode_splits(ATT_SPAN, items, most, (long)T * H * maps * (E + 2), scratch, scratch_floats);
  const int nw = items <= 256 && E < 256 ? 16 : (items <= 512 ? 8 : 4);
  const size_t lds = ((size_t)rh * D + (prep ? (size_t)(maps * D + E) / 2 : 0) + (size_t)nw * rh * E + (size_t)(nw + 1) * rh * 2) * sizeof(float);
#define ATT_GO_AS(RH, LPR, NW, MAPS, PREP, ARG)                                                                                       \
  do {                                                                                                                               \
    if (ensure_dynamic_lds<attn_decode_kernel<P, RH, LPR, NW, MAPS, false, PREP>>(lds) != UMB_OK) return UMB_EHIP;                    \
    hipLaunchKernelGGL((attn_decode_kernel<P, RH, LPR, NW, MAPS, false, PREP>), dim3(T, hblocks, nsplit), dim3(NW * 64), lds, st, (u16*)out, ldo, q, \
                       *kv, proj, ld, gate_col, bias, n_dist, pos, slot, H, G, D, window, scale, out_scale, softcap, form, scratch, nsplit, ARG); \
  } while (0)
#define ATT_GO(RH, LPR, NW, MAPS) do { if (prep) ATT_GO_AS(RH, LPR, NW, MAPS, true, *prep); else ATT_GO_AS(RH, LPR, NW, MAPS, false, DecodePrep{}); } while (0)
#define ATT_NW(RH, LPR, MAPS) do { if (nw == 16) ATT_GO(RH, (LPR < 32 ? LPR : 16), 16, MAPS); else if (nw == 8) ATT_GO(RH, LPR, 8, MAPS); else ATT_GO(RH, LPR, 4, MAPS); } while (0)
#define ATT_RH(LPR)                                                                                  \
  do {                                                                                               \
    if (maps == 2) { if (rh == 4) ATT_NW(4, LPR, 2); else ATT_NW(2, LPR, 2); }                        \
    else if (rh == 4) ATT_NW(4, LPR, 1); else if (rh == 2) ATT_NW(2, LPR, 1); else ATT_NW(1, LPR, 1); \
  } while (0)
  if (E == 64) ATT_RH(8);
  else if (E == 128) ATT_RH(16);
  else ATT_RH(32);
#undef ATT_RH
#undef ATT_NW
#undef ATT_GO
#undef ATT_GO_AS
  if (nsplit > 1) {
    if (maps == 2)
      hipLaunchKernelGGL((bsa_merge_kernel<P, 2>), dim3(T, H), dim3(64), 0, st, (u16*)out, ldo, scratch, proj, ld, gate_col, H, E, nsplit,
                         out_scale, form, pos, window);
    else
      hipLaunchKernelGGL((bsa_merge_kernel<P, 1>), dim3(T, H), dim3((unsigned)std::min(E + 63, 512) & ~63u), 0, st, (u16*)out, ldo, scratch, proj, ld, gate_col, H, E, nsplit,
                         out_scale, form, pos, window);
  }
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// The same for latent rows of 64, 128, 256 or 512 columns and rotary columns behind them, a multiple of 32 in all; false: another kernel's
static inline bool lat_decode_ok(int kv_rank, int rot_dim, int dtype, const UmbPagedKV* kv) {
  return dtype != UMB_SEQ_F32 && (kv_rank == 64 || kv_rank == 128 || kv_rank == 256 || kv_rank == 512) && (kv_rank + rot_dim) % 32 == 0 &&
         kv_rank + rot_dim <= 640 && (uintptr_t)kv->k % 16 == 0;
}
template <typename P, int RH, int LPR>
static int lat_decode_as(void* out, const float* qa, const UmbPagedKV* kv, const void* sink, const int* pos, const int* slot, int T, int H, int Dk, int window,
                         float scale, float* scratch, long scratch_floats, hipStream_t st) {
  constexpr int E = LPR * 8;
  const long items = (long)T * (H / RH);
  const int nsplit = decode_splits(LAT_SPAN, items, std::min((long)window, (long)kv->max_pages * kv->page), (long)T * H * (E + 2), scratch, scratch_floats);
  const int nw = nsplit > 1 ? 4 : items <= 256 && E < 256 ? 16 : (items <= 512 ? 8 : 4);
  const size_t lds = ((size_t)RH * Dk + (size_t)nw * RH * E + (size_t)(nw + 1) * RH * 2) * sizeof(float);
  const UmbAttnForm form{1, 0, reinterpret_cast<const float*>(sink), 0.f, 0.f, 0, 0};
#define LAT_GO(NW)                                                                                                                            \
  do {                                                                                                                                         \
    if (ensure_dynamic_lds<attn_decode_kernel<P, RH, LPR, NW, 1, true>>(lds) != UMB_OK) return UMB_EHIP;                                       \
    hipLaunchKernelGGL((attn_decode_kernel<P, RH, LPR, NW, 1, true>), dim3(T, H / RH, nsplit), dim3(NW * 64), lds, st, (u16*)out, H * E, qa, *kv, \
                       (const float*)nullptr, 0, -1, (const float*)nullptr, 0, pos, slot, H, 1, Dk, window, scale, 1.f, 0.f, form, scratch, nsplit, DecodePrep{}); \
  } while (0)
  if constexpr (E < 256) { if (nw == 16) LAT_GO(16); else if (nw == 8) LAT_GO(8); else LAT_GO(4); }
  else { if (nw == 8) LAT_GO(8); else LAT_GO(4); }
#undef LAT_GO
  if (nsplit > 1)
    hipLaunchKernelGGL((bsa_merge_kernel<P, 1, true>), dim3(T, H), dim3(std::min(E, 512)), 0, st, (u16*)out, H * E, scratch, (const float*)nullptr, 0, -1, H, E, nsplit, 1.f,
                       form, pos, window);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
// -1: not a shape of these
int lat_decode(void* out, const float* qa, const UmbPagedKV* kv, const void* sink, const int* pos, const int* slot, int T, int H, int kv_rank, int rot_dim,
               int window, float scale, float* scratch, long scratch_floats, int dtype, hipStream_t st) {
  if (!lat_decode_ok(kv_rank, rot_dim, dtype, kv)) return -1;
  const int Dk = kv_rank + rot_dim;
  const bool two = (long)T * H <= 128;                     // as in attn_decode
#define LAT_RH(LPR)                                                                                                                     \
  do {                                                                                                                                   \
    if (H % 4 == 0 && !two) return lat_decode_as<P, 4, LPR>(out, qa, kv, sink, pos, slot, T, H, Dk, window, scale, scratch, scratch_floats, st); \
    if (H % 2 == 0) return lat_decode_as<P, 2, LPR>(out, qa, kv, sink, pos, slot, T, H, Dk, window, scale, scratch, scratch_floats, st); \
    return lat_decode_as<P, 1, LPR>(out, qa, kv, sink, pos, slot, T, H, Dk, window, scale, scratch, scratch_floats, st);                 \
  } while (0)
  auto shape = [&](auto p) -> int {
    using P = decltype(p);
    if (kv_rank == 64) LAT_RH(8);
    if (kv_rank == 128) LAT_RH(16);
    if (kv_rank == 256) LAT_RH(32);
    LAT_RH(64);
  };
  return dtype == UMB_SEQ_BF16 ? shape(BF16{}) : shape(F16{});
#undef LAT_RH
}

extern "C" int umb_attn_attend(void* out, int ldo, const float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col,
                               const float* bias, int n_dist, const int* pos, const int* slot, int T, int H, int G, int D, int E,
                               int window, float scale, float out_scale, float softcap, const UmbAttnForm* form_, float* scratch,
                               long scratch_floats, int dtype, hipStream_t st) {
  if (T < 1 || H < 1 || G < 1 || H % G || D < 1 || E < 1 || E > 64 * BSA_MAXC || window < 1 || !out || !q || !bsa_kv_ok(kv) ||
      !pos || !slot || ldo < H * E || (bias && n_dist < 1) || !form_ok(form_))
    return UMB_EINVAL;
  const UmbAttnForm form = form_ ? *form_ : UmbAttnForm{1, 0, nullptr, 0.f, 0.f, 0, 0};
  if (gate_col >= 0 && (!proj || ld < gate_col + form_gate_cols(form, H, E))) return UMB_EINVAL;
  if (decode_rows_ok(D, E, dtype, kv)) {
    if (dtype == UMB_SEQ_BF16)
      return attn_decode<BF16>(out, ldo, q, kv, proj, ld, gate_col, bias, n_dist, pos, slot, T, H, G, D, E, window, scale, out_scale, softcap,
                               form, scratch, scratch_floats, st);
    return attn_decode<F16>(out, ldo, q, kv, proj, ld, gate_col, bias, n_dist, pos, slot, T, H, G, D, E, window, scale, out_scale, softcap,
                            form, scratch, scratch_floats, st);
  }
  const int maps = form.maps;
  const int hpg = H / G, nc = (E + 63) / 64;
  const int Dp = (D + 3) & ~3, Ep = (E + 3) & ~3, Mp = Dp > Ep ? Dp : Ep;
  // rows (head, map) of one workgroup: query heads of one key/value head, as many as divide the group and fit the register budget
  int rh = nc <= 2 ? 8 : (nc <= 4 ? 4 : 2);
  while (rh > maps && hpg % (rh / maps)) rh >>= 1;
  // A handful of (token, head block) items leaves most of the chip idle while each walks all its keys: with scratch for the
  // partial results the keys of an item are dealt to several workgroups (whole groups of four 64-key rounds by number, so the
  // order of every sum is a function of the position and of the step's row count only) and merged by a second launch.
  const int hblocks = H * maps / rh;
  const long items = (long)T * hblocks;
  int nsplit = 1;
  if (scratch && items <= 64) {                          // fewer than ~2048 waves in all with sixteen waves per item
    nsplit = (int)(512 / items) < 16 ? (int)(512 / items) : 16;
    // keys of one chunk or window only: no more workgroups than there can be groups of four rounds
    const long most = (long)(form.chunk > 0 && form.chunk < window ? form.chunk : window) + form.keep_first;
    if (nsplit > (most + 255) / 256) nsplit = (int)((most + 255) / 256);
    while (nsplit > 1 && (long)T * H * maps * nsplit * (E + 2) > scratch_floats) nsplit >>= 1;
  }
  const dim3 grid(T, hblocks, nsplit);
  int nw = (nsplit > 1 || items >= 1024) ? 4 : 16;
  auto lds_of = [&](int w) { return ((size_t)w * rh * Mp + (size_t)w * 2 * rh + (size_t)w * (rh * 64 + 128)) * sizeof(float); };
  if (nw == 16 && lds_of(16) > 128 * 1024) nw = 4;
  if (lds_of(nw) > 160 * 1024) return UMB_EINVAL;
  const size_t lds = lds_of(nw);
#define BSA_GO(RH, NC, NW, MAPS)                                                                                             \
  SEQ_TRY_((bsa_launch<P, RH, NC, NW, MAPS>(grid, lds, st, out, ldo, q, *kv, proj, ld, gate_col, bias, n_dist, pos, slot, H, G, D,   \
                                           E, window, scale, out_scale, softcap, form, scratch, nsplit)))
#define SEQ_TRY_(call) do { const int rc__ = (call); if (rc__ != UMB_OK) return rc__; } while (0)
#define BSA_NW(RH, NC, MAPS)                                                                                                 \
  do { if (nw == 16) BSA_GO(RH, NC, 16, MAPS); else BSA_GO(RH, NC, 4, MAPS); } while (0)
#define BSA_RH(NC)                                                                                                           \
  do {                                                                                                                       \
    if (maps == 2) { if (rh == 8) BSA_NW(8, NC, 2); else if (rh == 4) BSA_NW(4, NC, 2); else BSA_NW(2, NC, 2); }              \
    else if (rh == 8) BSA_NW(8, NC, 1); else if (rh == 4) BSA_NW(4, NC, 1); else if (rh == 2) BSA_NW(2, NC, 1);               \
    else BSA_NW(1, NC, 1);                                                                                                   \
  } while (0)
  DISPATCH_SEQ_DTYPE(dtype, {
    typedef typename El<P>::type El_;
    if (nc <= 1) BSA_RH(1);
    else if (nc <= 2) BSA_RH(2);
    else if (nc <= 4) {
      if (maps == 2) { if (rh == 4) BSA_NW(4, 4, 2); else BSA_NW(2, 4, 2); }
      else if (rh == 4) BSA_NW(4, 4, 1); else if (rh == 2) BSA_NW(2, 4, 1); else BSA_NW(1, 4, 1);
    } else {
      if (maps == 2) BSA_NW(2, 8, 2); else if (rh == 2) BSA_NW(2, 8, 1); else BSA_NW(1, 8, 1);
    }
    if (nsplit > 1) {
      if (maps == 2)
        hipLaunchKernelGGL((bsa_merge_kernel<P, 2>), dim3(T, H), dim3(64), 0, st, (El_*)out, ldo, scratch, proj, ld, gate_col, H, E,
                           nsplit, out_scale, form, pos, 0);
      else
        hipLaunchKernelGGL((bsa_merge_kernel<P, 1>), dim3(T, H), dim3((unsigned)std::min(E + 63, 512) & ~63u), 0, st, (El_*)out, ldo, scratch, proj, ld, gate_col, H, E,
                           nsplit, out_scale, form, pos, 0);
    }
  })
#undef BSA_RH
#undef BSA_NW
#undef BSA_GO
#undef SEQ_TRY_
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_attn_step(void* out, int ldo, float* q, const UmbPagedKV* kv, const float* proj, int ld, int append, const void* w_q, const void* w_k,
                             int norm_qk, int norm_v, const float* freq, int rot_dims, int layout, float rot_mult, float temp_coef, int temp_every, float eps,
                             const UmbValueMix* mix, int gate_col, const float* bias, int n_dist, const int* pos, const int* slot, int T, int H, int G,
                             int D, int E, int window, float scale, float out_scale, float softcap, const UmbAttnForm* form_, float* scratch,
                             long scratch_floats, int dtype, hipStream_t st) {
  const UmbAttnForm form = form_ ? *form_ : UmbAttnForm{1, 0, nullptr, 0.f, 0.f, 0, 0};
  if (!form_ok(form_) || !bsa_kv_ok(kv) || !out || !prep_ok(kv, proj, ld, append, pos, slot, freq, rot_dims, layout, T, H, G, D, E, form.maps) || window < 1 ||
      ldo < H * E || (bias && n_dist < 1) || (gate_col >= 0 && ld < gate_col + form_gate_cols(form, H, E)))
    return UMB_EINVAL;
  if (decode_rows_ok(D, E, dtype, kv)) {
    const DecodePrep prep{prep_of(append, norm_qk, norm_v, rot_dims, layout, rot_mult, H, G, D, E, form.maps, temp_coef, temp_every, eps, mix), w_q, w_k, freq};
    if (dtype == UMB_SEQ_BF16)
      return attn_decode<BF16>(out, ldo, nullptr, kv, proj, ld, gate_col, bias, n_dist, pos, slot, T, H, G, D, E, window, scale, out_scale, softcap, form,
                               scratch, scratch_floats, st, &prep);
    return attn_decode<F16>(out, ldo, nullptr, kv, proj, ld, gate_col, bias, n_dist, pos, slot, T, H, G, D, E, window, scale, out_scale, softcap, form,
                            scratch, scratch_floats, st, &prep);
  }
  const int rc = umb_attn_prep_mix(q, kv, proj, ld, append, w_q, w_k, norm_qk, norm_v, pos, slot, freq, rot_dims, layout, rot_mult, T, H, G, D, E, form.maps,
                                   temp_coef, temp_every, eps, mix, dtype, st);
  return rc != UMB_OK ? rc : umb_attn_attend(out, ldo, q, kv, proj, ld, gate_col, bias, n_dist, pos, slot, T, H, G, D, E, window, scale, out_scale, softcap,
                                             form_, scratch, scratch_floats, dtype, st);
}

extern "C" int umb_bsa_attend(void* out, int ldo, const float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col,
                              const float* bias, int n_dist, const int* pos, const int* slot, int T, int H, int G, int D, int E,
                              int window, float scale, float out_scale, float softcap, float* scratch, long scratch_floats,
                              int dtype, hipStream_t st) {
  return umb_attn_attend(out, ldo, q, kv, proj, ld, gate_col, bias, n_dist, pos, slot, T, H, G, D, E, window, scale, out_scale,
                         softcap, nullptr, scratch, scratch_floats, dtype, st);
}

// ---- prompt attention on the matrix pipe (16-bit storage; D a multiple of 8, E a multiple of 16).
// Workgroup = (16 consecutive positions of one sequence, one key/value head, four of its query heads), a wave per head.  The tile's
// keys -- from the first position's window start to the last position -- are walked in steps of 32 by the whole workgroup: the
// step's 32 cached key rows and value rows stand ONCE in LDS (seq_rows.h) and serve every head of the workgroup; the next step's
// are on their way to a second buffer while the current one is used.  Per step and head: two 16-key score tiles; the bias of the
// lane's eight (query, key) pairs, fetched by distance a step ahead; online softmax in fp32 with base-2
// exponents, accumulators rescaled only when a maximum moved; the lane's eight weights ARE its share of the B operand of the
// value product.  Scores and weights keep fp32 accuracy on the 16-bit pipe: the fp32 queries and the fp32 weights enter as
// high + low 16-bit halves (two products each, 2^-17 relative).
// Products per step at compile time: NSM steps of 32 features and NVM tiles of 16 columns, the least of a few sizes that hold D and E, with zeros
// behind a key row's D columns.  With run-time counts every product stood in a block of its own behind its own LDS read; with a whole step's
// reads free to move ahead, and steps that every query sees whole left untested, 1999 positions, 32 + 8 heads of 128 went from 212 us to 141, two
// maps over 617 positions, 64 | 128, from 104 to 71; rows by LDS-DMA, transposed reads in place of 2-byte stores, one barrier a step and fragments read
// ahead of their products: 117 and 59, two maps of 128 | 256 over 2000 positions 252 -> 182.
// What bounds it is vector instructions, half of which were addresses: 345 a step of 32 keys with a bias (32 products beside them).  Rows that fill
// their tile are fetched by a lane's own place plus constants (RowLanes: 76 -> 9 a step), a bias walks by distance (91 -> 32) and is asked for where the
// step before has used its own: with a bias 1999 positions, 32 + 8 heads of 128 159 us -> 136, of 64 116 -> 94, without 138 -> 123, two maps of
// 128 | 256 245 -> 213.  Held to four waves a SIMD the loop spills (36 registers of heads of 128): 211.
// FULL: D and E fill them, staging then tests nothing (2000 positions of 128: 158 us, 162 without).  us, run-time / these counts, 2000 positions: heads of 96 86 / 75, of 112 242 / 202, of 256 216 / 156, two maps of 128 | 128 273 / 179.
// Two heads a wave, sharing the value fragments, are behind wherever a launch is not several rounds of workgroups: 600 positions, 64 + 8 heads
// of 128 67 against 55, of 64 42 / 35 (2000 positions 195 / 198, 134 / 121).
constexpr float BSA_LOG2E = 1.4426950408889634f;

template <typename P> __device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo) {
  hi = pack2<P>(a, b);
  lo = pack2<P>(a - lo_f<P>(hi), b - hi_f<P>(hi));
}

// MAPS rows per wave, the maps of its head; every map has its part of the staged key rows, the value fragments of a step serve both
template <int NSM, int NVM, int MAPS> struct BsaTile {
  typedef RowTile<4 * NSM * MAPS> Keys;                         // a map's part of a key row is NSM steps wide
  typedef RowTile<2 * NVM> Values;
  static constexpr unsigned STEP = Keys::BYTES + Values::BYTES;
  static constexpr size_t LDS = 2 * STEP + 2 * 32 * sizeof(unsigned);
};
template <typename P, int NSM, int NVM, int MAPS, bool FULL>
__global__ __launch_bounds__(256) void bsa_attend_mfma_kernel(u16* __restrict__ out, int ldo, const float* __restrict__ q,
                                                              UmbPagedKV kv, const float* __restrict__ proj, int ld, int gate_col,
                                                              const float* __restrict__ bias, int n_dist,
                                                              const int* __restrict__ seq_slot, const int* __restrict__ seq_row0,
                                                              const int* __restrict__ seq_pos0, const int* __restrict__ seq_len,
                                                              int H, int G, int D, int E, int window, float scale, float out_scale,
                                                              float softcap, UmbAttnForm form) {
  extern __shared__ __attribute__((aligned(16))) u16 bsa_lds[];
  typedef BsaTile<NSM, NVM, MAPS> Tile;
  if constexpr (FULL) { D = NSM * 32; E = NVM * 16; }
  constexpr int HPW = MAPS;                           // rows of scores per wave
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, j = lane & 15, g4 = lane >> 4;
  const int DK = MAPS * D, nv = E >> 4, ncd = D >> 3, ncv = E >> 3;
  const unsigned lds0 = (unsigned)(size_t)(lds_char*)bsa_lds;          // two buffers of a step's key rows and value rows
  unsigned* tab = reinterpret_cast<unsigned*>(bsa_lds + Tile::STEP);   // [2][32]: where two steps' rows stand in the cache
  const int b = blockIdx.y;
  // How many keys a tile sees depends on its place in the chunk (or, without a window, in the sequence).  Workgroups that share a CU
  // are about 256 apart in launch order, which is the same tile of another head block: every other run of 256 takes the tiles from the
  // far end, so a CU's workgroups add up to about the same work.
  const int row = b + (int)gridDim.y * (int)blockIdx.z, run = gridDim.x < 256 ? 256 / gridDim.x : 1;
  const int tile = (row / run) & 1 ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;
  const int n = seq_len[b], q0 = tile * 16;
  if (q0 >= n) return;                                // the whole workgroup
  const int hpg = H / G, hblocks = (hpg + 3) / 4;
  const int g = blockIdx.z / hblocks;
  const int hl = blockIdx.z % hblocks * 4 + wave;     // the wave's head inside the group
  const bool active = hl < hpg;                       // a wave without one still stages rows and meets the barriers
  const int slot = seq_slot[b], row0 = seq_row0[b], pos0 = seq_pos0[b];
  const int nq = n - q0 < 16 ? n - q0 : 16;
  const int i_first = pos0 + q0, i_last = i_first + nq - 1;
  const bool q_ok = j < nq;
  const int i_j = i_first + (q_ok ? j : nq - 1);
  const long qrow = row0 + q0 + (q_ok ? j : nq - 1);
  int j_lo = i_first - window + 1 > 0 ? i_first - window + 1 : 0;
  int c_lo = 0;                                       // first position of the query's own chunk
  if (form.chunk > 0) {
    j_lo = max(j_lo, i_first / form.chunk * form.chunk);
    c_lo = i_j / form.chunk * form.chunk;
  }
  const int lo_all = max(i_last - window + 1, form.chunk > 0 ? i_last / form.chunk * form.chunk : 0);         // first position every query sees
  const int kept = min(form.keep_first, j_lo);        // first positions in front of the walk: step rows 0 .. kept - 1, then j_lo .. i_last
  const int j_off = j_lo - kept;
  const int total = kept + i_last - j_lo + 1;
  const float scale2 = scale * BSA_LOG2E;
  const u16* kbase = reinterpret_cast<const u16*>(kv.k);
  const u16* vbase = reinterpret_cast<const u16*>(kv.v);
  auto key_at = [&](int kx) { return kx < kept ? kx : j_off + kx; };
  auto row_pos = [&](int kx) { return key_at(min(kx, total - 1)); };            // behind the last key the last one again, masked
  RowLanes<4 * NSM * MAPS, 4> key_rows(kbase, wave, lane);
  RowLanes<2 * NVM, 4> value_rows(vbase, wave, lane);
  auto issue = [&](int st) __attribute__((always_inline)) {
    const unsigned to = lds0 + (unsigned)(st & 1) * Tile::STEP;
    if constexpr (FULL && key_rows.OK && value_rows.OK) {
      key_rows.issue(tab + (st & 1) * 32, to, wave);
      value_rows.issue(tab + (st & 1) * 32, to + Tile::Keys::BYTES, wave);
      return;
    }
    auto row_of = [&](int r) { return tab[(st & 1) * 32 + r]; };
    rows_issue<4 * NSM * MAPS, 4>(kbase, DK, to, wave, lane, row_of, [&](int c) {
      if (FULL && Tile::Keys::CH == 4 * NSM * MAPS) return c;
      const int mp = MAPS == 2 && c >= 4 * NSM ? 1 : 0, cc = c - mp * 4 * NSM;
      return cc < ncd ? mp * ncd + cc : -1;           // zeros past a map's D columns
    });
    rows_issue<2 * NVM, 4>(vbase, E, to + Tile::Keys::BYTES, wave, lane, row_of, [&](int c) { return (FULL && Tile::Values::CH == 2 * NVM) || c < ncv ? c : -1; });
  };
  const int hd = g * hpg + (active ? hl : hpg - 1);
  float bnext[8];
  auto ask_bias = [&](int base) __attribute__((always_inline)) {
    if (base >= kept) {                               // the walk itself: distances in a row from the lane's first one
      const int d0 = i_j - j_off - base - 4 * g4;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned at = 4u * (unsigned)min(max(d0 - 16 * (e >> 2) - (e & 3), 0), n_dist - 1);
        bnext[e] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(bias + (long)hd * n_dist) + at);
      }
      asm volatile("");                               // (or the loads are merged with those below, each with an address in two registers)
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int dd = i_j - key_at(base + 16 * (e >> 2) + 4 * g4 + (e & 3)), di = dd < 0 ? 0 : (dd < n_dist ? dd : n_dist - 1);
      bnext[e] = bias[(long)hd * n_dist + di];
    }
  };
  RowKeys<4 * NSM * MAPS> keys(j, g4);
  RowValues<2 * NVM> values(j, g4);
  const int steps = (total + 31) / 32;
  RowAsked next{};
  if (threadIdx.x < 64) tab[threadIdx.x] = pkv_tok_row(kv, slot, row_pos(threadIdx.x), g, G);
  if (threadIdx.x < 32) next.ask(kv, slot, row_pos(64 + threadIdx.x));
  if (bias) ask_bias(0);
  __syncthreads();
  issue(0);                                           // on its way beside the queries
  u32x4 qh[HPW][NSM], ql[HPW][NSM];
  f32x4 o[HPW][NVM];
  float m_run[HPW], l_run[HPW];
#pragma unroll
  for (int hh = 0; hh < HPW; ++hh) {
    const float* qr = q + ((qrow * H + hd) * MAPS + hh) * D;
#pragma unroll
    for (int s = 0; s < NSM; ++s) {
      const int d = 32 * s + 8 * g4;
      qh[hh][s] = u32x4{0u, 0u, 0u, 0u};
      ql[hh][s] = u32x4{0u, 0u, 0u, 0u};
      if (d < D) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(qr + d), c = *reinterpret_cast<const f32x4*>(qr + d + 4);
        unsigned hi[4], lo[4];
        split2<P>(a[0], a[1], hi[0], lo[0]);
        split2<P>(a[2], a[3], hi[1], lo[1]);
        split2<P>(c[0], c[1], hi[2], lo[2]);
        split2<P>(c[2], c[3], hi[3], lo[3]);
        qh[hh][s] = u32x4{hi[0], hi[1], hi[2], hi[3]};
        ql[hh][s] = u32x4{lo[0], lo[1], lo[2], lo[3]};
      }
    }
#pragma unroll
    for (int dt = 0; dt < NVM; ++dt) o[hh][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[hh] = -INFINITY;
    l_run[hh] = 0.f;
  }
  for (int st = 0; st < steps; ++st) {
    const int base = st * 32;
    // the step's rows have landed and nobody reads the step before any more: its buffer and its half of the table are free
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (threadIdx.x < 32) tab[(st & 1) * 32 + threadIdx.x] = next.row(kv, g, G);      // (in front of the issue: a wait for the look-up must not wait for that)
    if (st + 1 < steps) issue(st + 1);
    if (threadIdx.x < 32) next.ask(kv, slot, row_pos(base + 96 + threadIdx.x));
    if (!active) continue;
    keys.at_step(lds0 + (unsigned)(st & 1) * Tile::STEP);
    values.at_step(lds0 + (unsigned)(st & 1) * Tile::STEP + Tile::Keys::BYTES);
    // which of the lane's eight keys this query sees, and at what distance: the same for every head
    // (a step that every query sees whole needs no tests: rows past the last are not stored)
    const bool whole = base >= kept && j_off + base + 31 <= i_first && j_off + base >= lo_all;
    // fragments are read FR of them ahead of their products, the values' first ones in front of the softmax
    constexpr int FR = 4, NK = 2 * NSM * MAPS;
    u32x4 fr[FR];
    f32x4 sc2[HPW][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hh = 0; hh < HPW; ++hh) sc2[hh][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto key_frag = [&](int i) { return keys(i & 1, (i >> 1) % MAPS * NSM + (i >> 1) / MAPS); };         // (step of the map's features, map, key tile)
#pragma unroll
    for (int i = 0; i < FR; ++i) fr[i] = key_frag(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int u = i & 1, mp = (i >> 1) % MAPS, s = (i >> 1) / MAPS;
      sc2[mp][u] = P::mfma(fr[i % FR], ql[mp][s], sc2[mp][u]);
      sc2[mp][u] = P::mfma(fr[i % FR], qh[mp][s], sc2[mp][u]);
      fr[i % FR] = i + FR < NK ? key_frag(i + FR) : values(i + FR - NK);
      __builtin_amdgcn_sched_barrier(0);
    }
    u32x4 ph[HPW], pl[HPW];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
      // maxima and exponents in base 2 (scale2 = scale log2 e): one v_exp_f32 per weight
      float sv[8], mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) sv[e] = sc2[hh][e >> 2][e & 3] * scale2;
      if (softcap > 0.f) {                                           // (one test for all: eight of them stood between the products and the maximum)
#pragma unroll
        for (int e = 0; e < 8; ++e) sv[e] = softcap * tanhf(sc2[hh][e >> 2][e & 3] * scale / softcap) * BSA_LOG2E;      // capped, then to base 2
      }
      if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sv[e] += bnext[e] * BSA_LOG2E;
      }
      if (bias && hh == HPW - 1) ask_bias(base + 32);
      if (!whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int kx = base + 16 * (e >> 2) + 4 * g4 + (e & 3);
          const int jt = kx < kept ? kx : j_off + kx;
          sv[e] = q_ok && jt <= i_j && ((jt > i_j - window && jt >= c_lo) || jt < form.keep_first) ? sv[e] : -INFINITY;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sv[e]);
      const float m_new = fmaxf(m_run[hh], quad_max(mx));
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;          // a row that has seen no key yet: all weights 0
      const float fac = __builtin_amdgcn_exp2f(m_run[hh] - m_ref);
      float w[8], sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        w[e] = __builtin_amdgcn_exp2f(sv[e] - m_ref);
        sum += w[e];
      }
      l_run[hh] = l_run[hh] * fac + sum;                             // this lane's keys: added over the four lanes behind the walk
      m_run[hh] = m_new;
      if (__ballot(fac != 1.f)) {                                    // the maximum moved for some row of the tile
#pragma unroll
        for (int dt = 0; dt < NVM; ++dt) { o[hh][dt][0] *= fac; o[hh][dt][1] *= fac; o[hh][dt][2] *= fac; o[hh][dt][3] *= fac; }
      }
      unsigned hi[4], lo[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) split2<P>(w[2 * e], w[2 * e + 1], hi[e], lo[e]);
      ph[hh] = u32x4{hi[0], hi[1], hi[2], hi[3]};
      pl[hh] = u32x4{lo[0], lo[1], lo[2], lo[3]};
    }
    // O^T[d][query] += V^T[d][keys] P^T[keys][query]: lane (d row j of tile dt, quad g4) reads its 8 keys' values
#pragma unroll
    for (int dt = 0; dt < NVM; ++dt) {
#pragma unroll
      for (int hh = 0; hh < HPW; ++hh) {
        o[hh][dt] = P::mfma(fr[(dt + NK) % FR], pl[hh], o[hh][dt]);
        o[hh][dt] = P::mfma(fr[(dt + NK) % FR], ph[hh], o[hh][dt]);
      }
      if (dt + FR < NVM) fr[(dt + NK) % FR] = values(dt + FR);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int hh = 0; hh < HPW; ++hh) {
    l_run[hh] += __shfl_xor(l_run[hh], 16, 64);
    l_run[hh] += __shfl_xor(l_run[hh], 32, 64);
  }
  // lane holds O^T[d = 16 dt + 4 g4 + rr][query j]
  if (q_ok && active) {
    const bool gate_head = gate_col >= 0 && !form.gate_elem;
    const float gt = gate_head ? 1.f / (1.f + expf(-proj[qrow * ld + gate_col + hd])) : 1.f;
    const float* ge = gate_col >= 0 && form.gate_elem ? proj + qrow * ld + gate_col + (long)hd * E : nullptr;
    float l[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; ++mp) l[mp] = l_run[mp] + (form.sink ? __builtin_amdgcn_exp2f(form.sink[hd] * BSA_LOG2E - m_run[mp]) : 0.f);
    float inv = out_scale * gt / l[0];
    if constexpr (MAPS == 2) {                        // o = a1 - lambda a2 over the root mean square of the head's E columns
      const float i1 = 1.f / l[0], i2 = form.lambda / l[1];
      float ss = 0.f;
#pragma unroll
      for (int dt = 0; dt < NVM; ++dt) {
        if (dt < nv) {
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const float v = o[0][dt][rr] * i1 - o[1][dt][rr] * i2;
            o[0][dt][rr] = v;
            ss += v * v;
          }
        }
      }
      ss += __shfl_xor(ss, 16, 64);                   // the query's column quads: lanes j, j + 16, j + 32, j + 48 (all active)
      ss += __shfl_xor(ss, 32, 64);
      inv = out_scale * gt / sqrtf(ss / (float)E + form.eps);
    }
    u16* orow = out + qrow * ldo + (long)hd * E;
#pragma unroll
    for (int dt = 0; dt < NVM; ++dt) {
      if (dt < nv) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int d = 16 * dt + 4 * g4 + rr;
          float v = o[0][dt][rr] * inv;
          if (ge) v /= 1.f + expf(-ge[d]);
          orow[d] = P::from_f(v);
        }
      }
    }
  }
}

extern "C" int umb_bsa_attend_tiled_ok(int H, int G, int D, int E, int dtype) {
  return H >= 1 && G >= 1 && H % G == 0 && (dtype == UMB_SEQ_BF16 || dtype == UMB_SEQ_F16) && D >= 8 && D % 8 == 0 && D <= 256 &&
         E >= 16 && E % 16 == 0 && E <= 256;
}

extern "C" int umb_attn_attend_tiled(void* out, int ldo, const float* q, const UmbPagedKV* kv, const float* proj, int ld,
                                     int gate_col, const float* bias, int n_dist, const int* seq_slot, const int* seq_row0,
                                     const int* seq_pos0, const int* seq_len, int B, int max_len, int H, int G, int D, int E,
                                     int window, float scale, float out_scale, float softcap, const UmbAttnForm* form_, int dtype,
                                     hipStream_t st) {
  if (B < 1 || B > 65535 || max_len < 1 || window < 1 || !out || !q || !bsa_kv_ok(kv) || !seq_slot || !seq_row0 || !seq_pos0 ||
      !seq_len || ldo < H * E || (bias && n_dist < 1) || !umb_bsa_attend_tiled_ok(H, G, D, E, dtype) || !form_ok(form_))
    return UMB_EINVAL;
  if (!bias) n_dist = 1;
  const UmbAttnForm form = form_ ? *form_ : UmbAttnForm{1, 0, nullptr, 0.f, 0.f, 0, 0};
  if (gate_col >= 0 && (!proj || ld < gate_col + form_gate_cols(form, H, E))) return UMB_EINVAL;
  const int hpg = H / G, maps = form.maps;
#define BSA_MFMA_AS(NSM, NVM, MAPS, FULL)                                                                               \
  do {                                                                                                                     \
    const int hblocks = (hpg + 3) / 4;                                                                                     \
    if ((long)G * hblocks > 65535) return UMB_EINVAL;                                                                      \
    const dim3 grid((max_len + 15) / 16, B, G * hblocks);                                                                  \
    constexpr size_t lds = BsaTile<NSM, NVM, MAPS>::LDS;                                                                   \
    if (ensure_dynamic_lds<bsa_attend_mfma_kernel<P, NSM, NVM, MAPS, FULL>>(lds) != UMB_OK) return UMB_EHIP;          \
    hipLaunchKernelGGL((bsa_attend_mfma_kernel<P, NSM, NVM, MAPS, FULL>), grid, dim3(256), lds, st, (u16*)out, ldo, q, *kv, \
                       proj, ld, gate_col, bias, n_dist, seq_slot, seq_row0, seq_pos0, seq_len, H, G, D, E, window, scale, \
                       out_scale, softcap, form);                                                                          \
  } while (0)
#define BSA_MFMA(NSM, NVM, MAPS)                                                                                      \
  do { if (D == 32 * NSM && E == 16 * NVM) BSA_MFMA_AS(NSM, NVM, MAPS, true); else BSA_MFMA_AS(NSM, NVM, MAPS, false); } while (0)
#define BSA_MFMA_SHAPE()                                                                                                   \
  if (maps == 2) {                                                                                                         \
    if (D <= 64 && E <= 128) BSA_MFMA(2, 8, 2);                                                                         \
    else if (D <= 128 && E <= 128) BSA_MFMA(4, 8, 2);                                                                   \
    else if (D <= 128) BSA_MFMA(4, 16, 2);                                                                              \
    else BSA_MFMA(8, 16, 2);                                                                                            \
  } else if (D <= 64 && E <= 64) BSA_MFMA(2, 4, 1);                                                                     \
  else if (D <= 96 && E <= 96) BSA_MFMA(3, 6, 1);                                                                       \
  else if (D <= 128 && E <= 128) BSA_MFMA(4, 8, 1);                                                                     \
  else if (D <= 192 && E <= 192) BSA_MFMA(6, 12, 1);                                                                    \
  else BSA_MFMA(8, 16, 1)
  if (dtype == UMB_SEQ_BF16) { using P = BF16; BSA_MFMA_SHAPE(); }
  else { using P = F16; BSA_MFMA_SHAPE(); }
#undef BSA_MFMA_SHAPE
#undef BSA_MFMA_AS
#undef BSA_MFMA
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_bsa_attend_tiled(void* out, int ldo, const float* q, const UmbPagedKV* kv, const float* proj, int ld,
                                    int gate_col, const float* bias, int n_dist, const int* seq_slot, const int* seq_row0,
                                    const int* seq_pos0, const int* seq_len, int B, int max_len, int H, int G, int D, int E,
                                    int window, float scale, float out_scale, float softcap, int dtype, hipStream_t st) {
  return umb_attn_attend_tiled(out, ldo, q, kv, proj, ld, gate_col, bias, n_dist, seq_slot, seq_row0, seq_pos0, seq_len, B, max_len, H,
                               G, D, E, window, scale, out_scale, softcap, nullptr, dtype, st);
}
