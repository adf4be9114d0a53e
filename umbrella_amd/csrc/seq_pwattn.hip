// Sliding-window attention with mean-pooled blocks behind the window, sigmoid weights (no softmax, nothing normalised over
// keys), over a PAGED key/value store shared by many sequences.
//
//   position i sees   tokens j with 0 <= i - j < window
//              and    blocks b (positions b pool .. b pool + pool - 1) with b pool + pool - 1 <= i - window,
//                     each through ONE key = mean of its cached keys and ONE value = mean of its cached values;
//   tokens that left the window but whose block is not complete behind it are not seen at all.
//   weight of a visible key = sigmoid(q.k * scale + bias[head]);  out = sigmoid(gate) * sum weight * v.
//
// Keys are cached AFTER rotation and unit-RMS scaling, values are the key projection as it came out of the matrix product
// (before rotation and scaling): one projection serves both.  Rotary: interleaved pairs (2i, 2i+1) of the first rot_dims
// features turn by angle pos * freq[i], computed in fp32 with the full-range sincosf.
//
// Store: pages of `page` tokens handed out by the host-side manager; per layer K, V [pages][G][page][D] in the storage
// dtype and pooled K, V [pages][G][ceil(page / pool)][D] in fp32.  A pooled block lives in the page of its last position, so
// it is born complete (all its tokens are cached by then, in this or earlier pages of the sequence) and dies with the
// sequence.  The pooled mean is always taken over the cached (rounded) values in position order: the same numbers whether
// the tokens arrived in one step or one by one.
//
// Because the weights are not normalised there is no running maximum and no rescaling: a query's output is a plain sum.  A wave adds its
// rounds of keys in position order; how many waves share a query follows the launch (prompt tiles, or the number of (token, head block)
// items), so the same token in another batch, or of a prompt cut elsewhere, agrees to fp32 rounding and not bit for bit.
#include "seq_common.h"
#include "seq_decode.h"
#include "seq_rows.h"

// feature d (of D) of the sums of a pooled block's first cnt positions, keys and values, in order.  Lane j of a wave looks up position j's row, the rows go
// round as scalars and sixteen positions are in flight together.  Called by whole waves.
template <typename P>
__device__ __forceinline__ void pool_sums(const UmbPagedKV& kv, int slot, int first, int cnt, int g, int G, int D, int d, float& sk, float& sv) {
  typedef typename El<P>::type E;
  constexpr int KB = 16;
  const int lane = threadIdx.x & 63;
  for (int c = 0; c < cnt; c += 64) {
    const int some = cnt - c < 64 ? cnt - c : 64;
    const long off = pkv_tok(kv, slot, first + c + (lane < some ? lane : some - 1), g, G, D);
    for (int j0 = 0; j0 < some; j0 += KB) {
      E kk[KB], vv[KB];
#pragma unroll
      for (int u = 0; u < KB; ++u) {
        const int src = j0 + u < some ? j0 + u : some - 1;
        const unsigned lo = __builtin_amdgcn_readlane((unsigned)off, src), hi = __builtin_amdgcn_readlane((unsigned)(off >> 32), src);
        const long o = (long)(((unsigned long long)hi << 32) | lo) + d;
        kk[u] = reinterpret_cast<const E*>(kv.k)[o];
        vv[u] = reinterpret_cast<const E*>(kv.v)[o];
      }
#pragma unroll
      for (int u = 0; u < KB; ++u)
        if (j0 + u < some) {
          sk += ldf<P>(&kk[u]);
          sv += ldf<P>(&vv[u]);
        }
    }
  }
}

// one row of D features by a wave, turned and normed: put(d, value) for each, a pair a lane; raw(d, value) as projected
template <typename Raw, typename Put>
__device__ __forceinline__ void pwa_row(const float* __restrict__ src, int D, int rot_dims, const float* __restrict__ freq, int p, float eps, Raw raw, Put put) {
  const float pf = (float)p;
  const int lane = threadIdx.x & 63, pairs = (D + 1) / 2;
  auto turned = [&](int m, float& u, float& v) {
    if (2 * m + 1 < rot_dims) {
      float sn, cs;
      sincosf(pf * freq[m], &sn, &cs);
      const float ru = u * cs - v * sn, rv = v * cs + u * sn;
      u = ru; v = rv;
    }
  };
  // pass 1: rotate pairs, sum of squares (each lane owns whole pairs: features 2m, 2m+1 for m = lane, lane + 64, ...)
  float ss = 0.f;
  for (int m = lane; m < pairs; m += 64) {
    const int d0 = 2 * m, d1 = 2 * m + 1;
    float u = src[d0], v = d1 < D ? src[d1] : 0.f;
    raw(d0, u);
    if (d1 < D) raw(d1, v);
    turned(m, u, v);
    ss += u * u + (d1 < D ? v * v : 0.f);
  }
  ss = wave_sum(ss);
  const float f = 1.f / sqrtf(ss / (float)D + eps);
  for (int m = lane; m < pairs; m += 64) {
    const int d0 = 2 * m, d1 = 2 * m + 1;
    float u = src[d0], v = d1 < D ? src[d1] : 0.f;
    turned(m, u, v);
    put(d0, u * f);
    if (d1 < D) put(d1, v * f);
  }
}
// The same for the decode kernel: D features (a multiple of 32) as NP pairs a lane, asked for together with their frequencies in front of anything that
// waits, one angle a pair; compact, because what a launch executes once costs its fetch.  put(feature, turned, what norms it, as projected)
template <int D, typename Put>
__device__ __forceinline__ void pwa_row_few(const float* __restrict__ src, int rot_dims, const float* __restrict__ freq, int p, float eps, Put put) {
  constexpr int NP = (D + 127) / 128;
  typedef float pair __attribute__((ext_vector_type(2), aligned(4)));
  const int lane = threadIdx.x & 63;
  pair raw[NP];
  float u[NP], v[NP], fr[NP], ss = 0.f;
#pragma unroll
  for (int c = 0; c < NP; ++c) {
    const int m = min(lane + 64 * c, D / 2 - 1);
    raw[c] = *reinterpret_cast<const pair*>(src + 2 * m);
    fr[c] = 2 * m + 1 < rot_dims ? freq[m] : 0.f;
  }
#pragma unroll
  for (int c = 0; c < NP; ++c) {
    const int m = lane + 64 * c;
    u[c] = raw[c][0];
    v[c] = raw[c][1];
    if (2 * m + 1 < rot_dims) {
      float sn, cs;
      sincosf((float)p * fr[c], &sn, &cs);
      const float ru = fmaf(u[c], cs, -(v[c] * sn)), rv = fmaf(v[c], cs, u[c] * sn);
      u[c] = ru; v[c] = rv;
    }
    if (2 * m < D) ss += fmaf(u[c], u[c], fmaf(v[c], v[c], 0.f));
  }
  const float f = 1.f / sqrtf(wave_sum(ss) / (float)D + eps);
#pragma unroll
  for (int c = 0; c < NP; ++c) {
    const int m = lane + 64 * c;
    if (2 * m >= D) continue;
    put(2 * m, u[c], f, raw[c][0]);
    put(2 * m + 1, v[c], f, raw[c][1]);
  }
}
// the pooled block that the token at p completes, by a wave: the sums of the cached positions in front of it and its own key and value as they are stored
template <typename P>
__device__ __forceinline__ void pool_with(const UmbPagedKV& kv, int slot, const float* __restrict__ src, int g, int G, int D, int rot_dims,
                                          const float* __restrict__ freq, int p, float eps, int pool) {
  typedef typename El<P>::type E;
  const int lane = threadIdx.x & 63, blk = p / pool;
  const float pf = (float)p, inv = 1.f / (float)pool;
  float f = 0.f;
  {
    float ss = 0.f;
    for (int m = lane; m < (D + 1) / 2; m += 64) {
      const int d0 = 2 * m, d1 = 2 * m + 1;
      float u = src[d0], v = d1 < D ? src[d1] : 0.f;
      if (d1 < rot_dims) {
        float sn, cs;
        sincosf(pf * freq[m], &sn, &cs);
        const float ru = u * cs - v * sn, rv = v * cs + u * sn;
        u = ru; v = rv;
      }
      ss += u * u + (d1 < D ? v * v : 0.f);
    }
    f = 1.f / sqrtf(wave_sum(ss) / (float)D + eps);
  }
  const long dst = pkv_blk(kv, slot, blk, pool, g, G, D);
  for (int d0 = 0; d0 < D; d0 += 64) {                   // a feature a lane, and its partner's turn
    const int d = min(d0 + lane, D - 1), m = d >> 1, other = min(d ^ 1, D - 1);
    float sk = 0.f, sv = 0.f;
    pool_sums<P>(kv, slot, blk * pool, pool - 1, g, G, D, d, sk, sv);
    const float raw = src[d];
    float x = raw;
    if (2 * m + 1 < rot_dims) {
      float sn, cs;
      sincosf(pf * freq[m], &sn, &cs);
      x = d & 1 ? raw * cs + src[other] * sn : raw * cs - src[other] * sn;
    }
    E ks, vs;
    stf<P>(&ks, x * f);
    stf<P>(&vs, raw);
    sk += ldf<P>(&ks);
    sv += ldf<P>(&vs);
    if (d0 + lane < D) {
      kv.kp[dst + d] = sk * inv;
      kv.vp[dst + d] = sv * inv;
    }
  }
}

// ---- rotary + unit RMS + cache append.  One wave per (token, head slot); head slots 0..H-1 are queries, H..H+G-1 keys.
// pool > 0 (one token a sequence): slots H+G..H+2G-1 are the pooled blocks that the token completes, if it does: the sums of the cached positions in front of
// it and its own key and value, worked out once more, as they are stored.  us, in a launch of their own (pwa_pool_kernel, below) / here: 16 requests 4.7 + 4.6 -> 7.0,
// whether one completes a block or not; one request 4.1 + 1.8 -> 4.2.  Their loads in front of the rest: 7.4.
template <typename P>
__global__ __launch_bounds__(256) void pwa_prep_kernel(float* __restrict__ q, UmbPagedKV kv, const float* __restrict__ proj, int ld,
                                                       const int* __restrict__ pos, const int* __restrict__ slot,
                                                       const float* __restrict__ freq, int T, int H, int G, int D, int rot_dims,
                                                       float eps, int pool) {
  typedef typename El<P>::type E;
  const int wave = threadIdx.x >> 6, per = H + G + (pool > 0 ? G : 0);
  const long id = (long)blockIdx.x * 4 + wave;
  if (id >= (long)T * per) return;
  const int t = __builtin_amdgcn_readfirstlane((int)(id / per)), hs = __builtin_amdgcn_readfirstlane((int)(id % per));
  const bool is_q = hs < H, is_pool = hs >= H + G;
  const int g = is_q ? 0 : is_pool ? hs - H - G : hs - H, p = pos[t];
  const float* src = proj + (long)t * ld + (is_q ? (long)hs * D : (long)(H + g) * D);
  if (is_pool) {
    if ((p + 1) % pool == 0) pool_with<P>(kv, slot[t], src, g, G, D, rot_dims, freq, p, eps, pool);
    return;
  }
  if (is_q) {
    float* qd = q + (long)t * H * D + (long)hs * D;
    pwa_row(src, D, rot_dims, freq, p, eps, [](int, float) {}, [&](int d, float v) { qd[d] = v; });
    return;
  }
  const long off = pkv_tok(kv, slot[t], p, g, G, D);
  E* kd = reinterpret_cast<E*>(kv.k) + off;
  E* vd = reinterpret_cast<E*>(kv.v) + off;
  pwa_row(src, D, rot_dims, freq, p, eps, [&](int d, float v) { stf<P>(vd + d, v); }, [&](int d, float v) { stf<P>(kd + d, v); });
}

// The same for many items (heads of at most 128, an even number): a wave takes four neighbouring head slots of one token, reads them once,
// all loads in flight, and works the angles out once for the four.  Two passes of one slot each, both with their sines: 2048 tokens of
// 32 + 8 slots of 64 36 us, now 19.3.
template <typename P>
__global__ __launch_bounds__(256) void pwa_prep_four_kernel(float* __restrict__ q, UmbPagedKV kv, const float* __restrict__ proj, int ld,
                                                            const int* __restrict__ pos, const int* __restrict__ slot,
                                                            const float* __restrict__ freq, int T, int H, int G, int D, int rot_dims,
                                                            float eps, int groups) {
  typedef typename El<P>::type E;
  const int item = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6))), lane = threadIdx.x & 63;
  const int t = item / groups, s0 = item % groups * 4, d = 2 * lane;
  if (t >= T) return;
  const int p = pos[t], sl = slot[t];
  const bool ok = d < D, turn = d + 1 < rot_dims;
  float u[4], v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float* src = proj + (long)t * ld + (long)min(s0 + k, H + G - 1) * D;
    u[k] = ok ? src[d] : 0.f;
    v[k] = ok ? src[d + 1] : 0.f;
  }
  float sn = 0.f, cs = 1.f;
  if (turn) sincosf((float)p * freq[lane], &sn, &cs);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int hs = s0 + k;
    if (hs >= H + G) return;
    const bool is_q = hs < H;
    long off = 0;
    if (!is_q) {
      off = pkv_tok(kv, sl, p, hs - H, G, D) + d;
      if (ok) { stf<P>(reinterpret_cast<E*>(kv.v) + off, u[k]); stf<P>(reinterpret_cast<E*>(kv.v) + off + 1, v[k]); }
    }
    float a = u[k], b = v[k];
    if (turn) { a = u[k] * cs - v[k] * sn; b = v[k] * cs + u[k] * sn; }
    const float f = 1.f / sqrtf(wave_sum(a * a + b * b) / (float)D + eps);
    if (!ok) continue;
    if (is_q) {
      float* qd = q + ((long)t * H + hs) * D + d;
      qd[0] = a * f;
      qd[1] = b * f;
    } else {
      stf<P>(reinterpret_cast<E*>(kv.k) + off, a * f);
      stf<P>(reinterpret_cast<E*>(kv.k) + off + 1, b * f);
    }
  }
}

// The same where rows are 64 or 128 long and turned in whole quads: a wave takes PREP_QUADS quads a lane of one token's neighbouring slots, two or four side
// by side, all loads in flight, the angles worked out once for all of them; bound by its bytes, where four slots a wave were by their vector work (seq_battn.hip): 2048 tokens,
// 32 + 8 slots of 64 18.9 -> 10.8 us (10.2 with the sums of squares in another order than that kernel's).
constexpr int PREP_QUADS = 4;
constexpr int prep_rows(int D) { return PREP_QUADS * 256 / D; }      // slots a wave takes
template <typename P, int D>
__global__ __launch_bounds__(256) void pwa_prep_quads_kernel(float* __restrict__ q, UmbPagedKV kv, const float* __restrict__ proj, int ld,
                                                             const int* __restrict__ pos, const int* __restrict__ slot,
                                                             const float* __restrict__ freq, int T, int H, int G, int rot_dims, float eps, int waves) {
  typedef typename El<P>::type E;
  typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
  const int item = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6))), lane = threadIdx.x & 63;
  const int t = item / waves, first = (item - t * waves) * prep_rows(D), n = min(prep_rows(D), H + G - first);
  if (t >= T) return;
  const int p = pos[t], sl = slot[t], sub = lane / (D / 4), e = lane % (D / 4) * 4;
  f32x4 x[PREP_QUADS];
#pragma unroll
  for (int k = 0; k < PREP_QUADS; ++k) x[k] = *reinterpret_cast<const quad*>(proj + (long)t * ld + (first + min(k * (256 / D) + sub, n - 1)) * D + e);
  float sn[2] = {0.f, 0.f}, cs[2] = {1.f, 1.f};
  if (e < rot_dims) {
    float f0 = freq[e / 2], f1 = freq[e / 2 + 1];
#pragma unroll 1
    for (int i = 0; i < 2; ++i) {                          // one place for the sines, the values go round
      sn[0] = sn[1];
      cs[0] = cs[1];
      sincosf((float)p * f0, &sn[1], &cs[1]);
      f0 = f1;
    }
  }
  const long kv0 = pkv_tok(kv, sl, p, 0, G, D) + e;
#pragma unroll
  for (int k = 0; k < PREP_QUADS; ++k) {
    const int r = k * (256 / D) + sub, hs = first + min(r, n - 1);
    f32x4 o = x[k];
    if (e < rot_dims) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        o[2 * i] = fmaf(x[k][2 * i], cs[i], -(x[k][2 * i + 1] * sn[i]));
        o[2 * i + 1] = fmaf(x[k][2 * i + 1], cs[i], x[k][2 * i] * sn[i]);
      }
    }
    float sq[2];                                             // pairs, in the order of a wave with a pair a lane
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      sq[i] = fmaf(o[2 * i], o[2 * i], fmaf(o[2 * i + 1], o[2 * i + 1], 0.f));
      if constexpr (D == 128) {
        float b = sq[i];
        swap16(sq[i], b);
        sq[i] += b;
      }
      sq[i] = row_add16(sq[i]);
    }
    const float f = 1.f / sqrtf((sq[0] + sq[1]) / (float)D + eps);
    if (r >= n) continue;
    o = rounded(o * f);
    if (hs < H) *reinterpret_cast<f32x4*>(q + ((long)t * H + hs) * D + e) = o;
    else {
      const long off = kv0 + (long)(hs - H) * kv.page * D;
      st4<P>(reinterpret_cast<E*>(kv.k) + off, o);
      st4<P>(reinterpret_cast<E*>(kv.v) + off, x[k]);
    }
  }
}

// ---- pooled blocks completed by this step: grid (block-in-step, sequence, kv head), a thread per feature.
// Latency: a handful of workgroups, each a chain of page lookups and loads (pool_sums; one position at a time, each behind its own lookup, 16 positions
// took 19.3 us, now 4.4).
template <typename P>
__global__ __launch_bounds__(256) void pwa_pool_kernel(UmbPagedKV kv, const int* __restrict__ seq_slot,
                                                       const int* __restrict__ seq_pos0, const int* __restrict__ seq_len, int G,
                                                       int D, int pool) {
  const int b = blockIdx.y, g = blockIdx.z, lane = threadIdx.x & 63;
  const int p0 = seq_pos0[b], n = seq_len[b];
  if (n <= 0) return;
  // blocks whose last position e = blk pool + pool - 1 lies in [p0, p0 + n): blk >= ceil((p0 - pool + 1) / pool) = p0 / pool
  const int first = p0 / pool;
  const int blk = first + blockIdx.x;
  const int e = blk * pool + pool - 1;
  if (e >= p0 + n) return;
  const int slot = seq_slot[b];
  const long dst = pkv_blk(kv, slot, blk, pool, g, G, D);
  const float inv = 1.f / (float)pool;
  for (int d0 = threadIdx.x - lane; d0 < D; d0 += blockDim.x) {           // uniform in a wave
    const int d = d0 + lane < D ? d0 + lane : D - 1;
    float sk = 0.f, sv = 0.f;
    pool_sums<P>(kv, slot, blk * pool, pool, g, G, D, d, sk, sv);
    if (d0 + lane < D) {
      kv.kp[dst + d] = sk * inv;
      kv.vp[dst + d] = sv * inv;
    }
  }
}

// ---- attention.  Workgroup = (token, RH query heads of one key/value group): the heads of a group read the same keys and
// values, so one pass over the keys serves all of them.  The NW waves take the 64-key rounds w, w + NW, ... of the key list
// (pooled blocks first, then the window's tokens, both in position order) and their partial sums are added through LDS in
// wave order: which keys land in which wave depends on the query's position and on NW.  Score phase: lane = key, 16-byte loads along
// the key's row against the queries held in LDS.  Value phase: lane = value column, the round's weights broadcast one key at a time.
constexpr int PWA_MAXC = 4;      // value columns per lane: D <= 256

template <typename P, int RH, int NC, int NW>
__global__ __launch_bounds__(NW * 64) void pwa_attend_kernel(typename El<P>::type* __restrict__ out, const float* __restrict__ q,
                                                         UmbPagedKV kv, const float* __restrict__ proj, int ld, int gate_col,
                                                         const typename El<P>::type* __restrict__ pos_bias,
                                                         const int* __restrict__ pos, const int* __restrict__ slot_, int T, int H,
                                                         int G, int D, int window, int pool, float scale) {
  typedef typename El<P>::type E;
  extern __shared__ float lds[];
  constexpr int PWA_KB = 8;   // keys whose value rows are in flight together (32 measured 3x slower at 16 waves: registers)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int Dp = (D + 3) & ~3;
  float* q_s = lds;                                          // [RH][Dp] queries; later [NW][RH][Dp] partial outputs
  float* w_s = lds + NW * RH * Dp + wave * (RH * 64 + 128);  // per wave: [RH][64] weights, [64] 64-bit offsets
  long* off_s = reinterpret_cast<long*>(w_s + RH * 64);
  const int t = blockIdx.x, h0 = blockIdx.y * RH;
  const int g = h0 / (H / G);
  const int i = pos[t], slot = slot_[t];
  for (int x = threadIdx.x; x < RH * D; x += NW * 64) q_s[(x / D) * Dp + x % D] = q[(long)t * H * D + (long)h0 * D + x];
  float bias[RH];
#pragma unroll
  for (int r = 0; r < RH; ++r) bias[r] = pos_bias ? ldf<P>(pos_bias + h0 + r) : 0.f;
  __syncthreads();
  const int j_lo = i - window + 1 > 0 ? i - window + 1 : 0;
  const int n_blk = i - window + 1 >= pool ? (i - window + 1) / pool : 0;
  const int n_keys = n_blk + (i - j_lo + 1);
  const bool vec = (D & 7) == 0;
  float acc[RH][NC];
#pragma unroll
  for (int r = 0; r < RH; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[r][c] = 0.f;
  for (int base = wave * 64; base < n_keys; base += NW * 64) {
    const int kx = base + lane;
    float s[RH];
#pragma unroll
    for (int r = 0; r < RH; ++r) s[r] = 0.f;
    long off = 0;
    bool pooled = false;
    if (kx < n_keys) {
      pooled = kx < n_blk;
      off = pooled ? pkv_blk(kv, slot, kx, pool, g, G, D) : pkv_tok(kv, slot, j_lo + (kx - n_blk), g, G, D);
      if (pooled) {
        const float* kr = kv.kp + off;
        if ((D & 3) == 0) {
          for (int d = 0; d < D; d += 32) {              // eight 16-byte loads in flight, then their 32 x RH products
            f32x4 kk[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) kk[u] = *reinterpret_cast<const f32x4*>(kr + (d + 4 * u < D ? d + 4 * u : 0));
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              if (d + 4 * u >= D) break;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int r = 0; r < RH; ++r) s[r] += q_s[r * Dp + d + 4 * u + e] * kk[u][e];
              }
            }
          }
        } else {
          for (int d = 0; d < D; ++d) {
            const float kd = kr[d];
#pragma unroll
            for (int r = 0; r < RH; ++r) s[r] += q_s[r * Dp + d] * kd;
          }
        }
      } else {
        const E* kr = reinterpret_cast<const E*>(kv.k) + off;
        bool done = false;
        if constexpr (sizeof(E) == 2) {
          if (vec) {
            for (int d = 0; d < D; d += 64) {            // eight 16-byte loads in flight, then their 64 x RH products
              u32x4 kk[8];
#pragma unroll
              for (int u = 0; u < 8; ++u) kk[u] = *reinterpret_cast<const u32x4*>(kr + (d + 8 * u < D ? d + 8 * u : 0));
#pragma unroll
              for (int u = 0; u < 8; ++u) {
                if (d + 8 * u >= D) break;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const float k0 = lo_f<P>(kk[u][e]), k1 = hi_f<P>(kk[u][e]);
                  const int dd = d + 8 * u + 2 * e;
#pragma unroll
                  for (int r = 0; r < RH; ++r) s[r] += q_s[r * Dp + dd] * k0 + q_s[r * Dp + dd + 1] * k1;
                }
              }
            }
            done = true;
          }
        }
        if (!done) {
          for (int d = 0; d < D; ++d) {
            const float kd = ldf<P>(kr + d);
#pragma unroll
            for (int r = 0; r < RH; ++r) s[r] += q_s[r * Dp + d] * kd;
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RH; ++r) w_s[r * 64 + lane] = kx < n_keys ? 1.f / (1.f + expf(-(s[r] * scale + bias[r]))) : 0.f;
    off_s[lane] = pooled ? ~off : off;            // pooled entries are flagged by the complement (off >= 0 always)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int cnt = n_keys - base < 64 ? n_keys - base : 64;
    // value rows: PWA_KB keys are fetched together, then used.  The round's keys are pooled entries first (fp32), then
    // tokens (storage dtype): two loops, so that no load sits behind a branch on the entry's kind; indices past the end are
    // clamped and weighted 0.
    const int cntp = n_blk - base < 0 ? 0 : (n_blk - base < cnt ? n_blk - base : cnt);
    int dcl[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) dcl[c] = lane + 64 * c < D ? lane + 64 * c : D - 1;
    for (int j0 = 0; j0 < cntp; j0 += PWA_KB) {
      float vv[PWA_KB][NC];
#pragma unroll
      for (int u = 0; u < PWA_KB; ++u) {
        const long oj = ~off_s[j0 + u < cntp ? j0 + u : cntp - 1];
#pragma unroll
        for (int c = 0; c < NC; ++c) vv[u][c] = kv.vp[oj + dcl[c]];
      }
#pragma unroll
      for (int u = 0; u < PWA_KB; ++u) {
#pragma unroll
        for (int r = 0; r < RH; ++r) {
          const float wj = j0 + u < cntp ? w_s[r * 64 + j0 + u] : 0.f;
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[r][c] += wj * vv[u][c];
        }
      }
    }
    for (int j0 = cntp; j0 < cnt; j0 += PWA_KB) {
      float vv[PWA_KB][NC];
#pragma unroll
      for (int u = 0; u < PWA_KB; ++u) {
        const long oj = off_s[j0 + u < cnt ? j0 + u : cnt - 1];
#pragma unroll
        for (int c = 0; c < NC; ++c) vv[u][c] = ldf<P>(reinterpret_cast<const E*>(kv.v) + oj + dcl[c]);
      }
#pragma unroll
      for (int u = 0; u < PWA_KB; ++u) {
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
  for (int r = 0; r < RH; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = lane + 64 * c;
      if (d < D) lds[(wave * RH + r) * Dp + d] = acc[r][c];
    }
  __syncthreads();
  for (int x = threadIdx.x; x < RH * D; x += NW * 64) {
    const int r = x / D, d = x % D;
    float o = lds[(0 * RH + r) * Dp + d];
#pragma unroll
    for (int w = 1; w < NW; ++w) o += lds[(w * RH + r) * Dp + d];
    const float gate = 1.f / (1.f + expf(-proj[(long)t * ld + gate_col + h0 + r]));
    stf<P>(out + (long)t * H * D + (long)(h0 + r) * D + d, o * gate);
  }
}

// ---- attention of single tokens (see seq_decode.h; D = 64, 128 or 256 in 16-bit storage): rounds of 16 pooled entries, then rounds of 16
// tokens, dealt to the workgroup's waves; weights need no maximum, so the waves' sums are simply added.
// Before -> now, replayed from a graph, D 128: one token behind 40 / 2000 keys 10.7 -> 4.9 / 30.8 -> 18.0 us, 48 tokens behind 40 20.9 -> 5.7,
// 64 behind 1000 77 -> 45.
// PREP: steps of one token a sequence, as in seq_battn.hip: the queries come from the projection, the token's key and value stand in LDS for the round that
// needs them, and the group's first workgroup appends them and the block that they complete.  Compact, as there: 16 tokens, heads of 128,
// 11.0 -> 10.4 us inside a step.
struct PwaPrep { const float* freq; int rot_dims; float eps; };
template <typename P, int RH, int LPR, int NW, bool PREP>
__global__ __launch_bounds__(NW * 64) void pwa_decode_kernel(u16* __restrict__ out, const float* __restrict__ q, UmbPagedKV kv,
                                                             const float* __restrict__ proj, int ld, int gate_col,
                                                             const u16* __restrict__ pos_bias, const int* __restrict__ pos,
                                                             const int* __restrict__ slot_, int H, int G, int Dr, int window, int pool,
                                                             float scale, PwaPrep prep) {
  constexpr int D = LPR * 8, KPI = 64 / LPR, VL = 16 / KPI;      // Dr = D, but not at compile time: or a round's queries are all read ahead
  __shared__ __attribute__((aligned(16))) float q_s[RH * D];
  __shared__ __attribute__((aligned(16))) u16 new_k[PREP ? D : 8], new_v[PREP ? D : 8];
  extern __shared__ float o_s[];                           // [NW][RH][D]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 15, quarter = lane >> 4;
  const int t = blockIdx.x, h0 = blockIdx.y * RH, g = h0 / (H / G);
  const int i = pos[t], slot = slot_[t];
  const int j_lo = i - window + 1 > 0 ? i - window + 1 : 0;
  const int n_blk = i - window + 1 >= pool ? (i - window + 1) / pool : 0;
  const int n_tok = i - j_lo + 1, br = (n_blk + 15) / 16, rounds = br + (n_tok + 15) / 16;
  const int nact = min(NW, rounds);
  auto row_of = [&](int rd) {
    return rd < br ? pkv_blk_row(kv, slot, min(rd * 16 + j, n_blk - 1), pool, g, G)
                   : pkv_tok_row(kv, slot, j_lo + min((rd - br) * 16 + j, n_tok - 1), g, G);
  };
  unsigned row = 0;
  if (wave < nact) row = row_of(wave);
  // The first round's rows are on their way while the token's own are prepared, where it is the only round, as in seq_battn.hip, and a unit has one workgroup
  // (us a launch inside a step, without / with: 16 tokens, heads of 128 10.7 / 10.4; 128 tokens from a warm cache 15.9 / 17.6)
  unsigned near_k = 0, near_v = 0;
  if (PREP && NW == 16 && rounds <= NW && wave < nact) {
    const long eb = wave < br ? 4 : 2, at = (long)row * D + quarter * (D / 4);
    near_k = *reinterpret_cast<const unsigned*>(reinterpret_cast<const char*>(wave < br ? (const void*)kv.kp : kv.k) + at * eb);
    near_v = *reinterpret_cast<const unsigned*>(reinterpret_cast<const char*>(wave < br ? (const void*)kv.vp : kv.v) + at * eb);
  }
  if constexpr (PREP) {
    const float* src = proj + (long)t * ld;
    const bool append = h0 % (H / G) == 0;
#pragma unroll 1
    for (int task = wave; task < RH + 2; task += NW) {     // a row a wave
      if (task <= RH) {
        const bool is_q = task < RH;
        const long off = is_q ? 0 : pkv_tok(kv, slot, i, g, G, D);
        u16* kd = reinterpret_cast<u16*>(kv.k) + off;
        u16* vd = reinterpret_cast<u16*>(kv.v) + off;
        pwa_row_few<D>(src + (is_q ? h0 + task : H + g) * D, prep.rot_dims, prep.freq, i, prep.eps, [&](int d, float x, float f, float raw) {
          if (is_q) {
            q_s[task * D + d] = x * f;
            return;
          }
          const u16 kb = product_once<P>(x, f), vb = P::from_f(raw);
          new_k[d] = kb;
          new_v[d] = vb;
          if (append) { kd[d] = kb; vd[d] = vb; }
        });
      } else if (append && (i + 1) % pool == 0)
        pool_with<P>(kv, slot, src + (H + g) * D, g, G, Dr, prep.rot_dims, prep.freq, i, prep.eps, pool);
    }
  } else {
    for (int x = threadIdx.x; x < RH * D; x += NW * 64) q_s[x] = q[((long)t * H + h0) * D + x];
  }
  float bias[RH];
#pragma unroll
  for (int r = 0; r < RH; ++r) bias[r] = pos_bias ? P::to_f(pos_bias[h0 + r]) : 0.f;
  __syncthreads();
  if (wave < nact) {
    if (PREP && NW == 16) asm volatile("" :: "v"(near_k), "v"(near_v));      // (asked for, whatever they hold; no registers in the rounds)
    float acc[RH * 8];
#pragma unroll
    for (int v = 0; v < RH * 8; ++v) acc[v] = 0.f;
    float s[RH];
    auto dots = [&](const float* kf, int d) {
      const int at = d + quarter * 8;
#pragma unroll
      for (int r = 0; r < RH; ++r) {
        const f32x4 qa = *reinterpret_cast<const f32x4*>(q_s + r * D + at);
        const f32x4 qb = *reinterpret_cast<const f32x4*>(q_s + r * D + at + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[r] += qa[e] * kf[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[r] += qb[e] * kf[4 + e];
      }
    };
    auto weights = [&](bool valid) {
#pragma unroll
      for (int r = 0; r < RH; ++r) s[r] = valid ? 1.f / (1.f + expf(-(add_rows(s[r]) * scale + bias[r]))) : 0.f;
    };
    auto values = [&](const float* vf, int u) {
#pragma unroll
      for (int r = 0; r < RH; ++r) {
        const float w = __shfl(s[r], KPI * u + lane / LPR, 64);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r * 8 + e] += w * vf[e];
      }
    };
    int rd = wave;
    for (; rd < br; rd += NW) {                            // two loops: joined in one they need twice the registers
      const unsigned next_row = rd + NW < rounds ? row_of(rd + NW) : 0;
#pragma unroll
      for (int r = 0; r < RH; ++r) s[r] = 0.f;
      const float* kr = kv.kp + (long)row * D + quarter * 8;
      const float* vc = kv.vp + (lane & (LPR - 1)) * 8;
      for (int d = 0; d < Dr; d += 128) {
        f32x4 ka[4], kb[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float* kd = kr + (d + 32 * u < Dr ? d + 32 * u : 0);
          ka[u] = *reinterpret_cast<const f32x4*>(kd);
          kb[u] = *reinterpret_cast<const f32x4*>(kd + 4);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (d + 32 * u >= Dr) break;
          const float kf[8] = {ka[u][0], ka[u][1], ka[u][2], ka[u][3], kb[u][0], kb[u][1], kb[u][2], kb[u][3]};
          dots(kf, d + 32 * u);
        }
      }
      weights(rd * 16 + j < n_blk);
      // fp32 rows are twice as long as a token's: their values are fetched behind the scores, in registers that held the keys
      constexpr int VB = VL < 4 ? VL : 4;
#pragma unroll 1
      for (int u0 = 0; u0 < VL; u0 += VB) {
        f32x4 va[VB], vb[VB];
#pragma unroll
        for (int u = 0; u < VB; ++u) {
          const float* vr = vc + (long)(unsigned)__shfl((int)row, KPI * (u0 + u) + lane / LPR, 64) * D;
          va[u] = *reinterpret_cast<const f32x4*>(vr);
          vb[u] = *reinterpret_cast<const f32x4*>(vr + 4);
        }
#pragma unroll
        for (int u = 0; u < VB; ++u) {
          const float vf[8] = {va[u][0], va[u][1], va[u][2], va[u][3], vb[u][0], vb[u][1], vb[u][2], vb[u][3]};
          values(vf, u0 + u);
        }
      }
      row = next_row;
    }
    for (; rd < rounds; rd += NW) {
      const unsigned next_row = rd + NW < rounds ? row_of(rd + NW) : 0;
#pragma unroll
      for (int r = 0; r < RH; ++r) s[r] = 0.f;
      const u16* kr = reinterpret_cast<const u16*>(kv.k) + (long)row * D + quarter * 8;
      const u16* vc = reinterpret_cast<const u16*>(kv.v) + (lane & (LPR - 1)) * 8;
      u32x4 vv[VL];
#pragma unroll
      for (int u = 0; u < VL; ++u) vv[u] = *reinterpret_cast<const u32x4*>(vc + (long)(unsigned)__shfl((int)row, KPI * u + lane / LPR, 64) * D);
      // the round with the token's own key: it and the lanes behind it (whose weights are 0) take what LDS has, the cache does not have it yet
      const int key0 = (rd - br) * 16;
      const bool own = PREP && key0 + 16 >= n_tok;
      if (own) {
#pragma unroll
        for (int u = 0; u < VL; ++u)
          if (key0 + KPI * u + lane / LPR >= n_tok - 1) vv[u] = *reinterpret_cast<const u32x4*>(new_v + (lane & (LPR - 1)) * 8);
      }
#pragma unroll 1
      for (int d = 0; d < Dr; d += 128) {
        u32x4 kk[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) kk[u] = *reinterpret_cast<const u32x4*>(kr + (d + 32 * u < Dr ? d + 32 * u : 0));
        if (own && key0 + j >= n_tok - 1) {
#pragma unroll
          for (int u = 0; u < 4; ++u) kk[u] = *reinterpret_cast<const u32x4*>(new_k + (d + 32 * u < Dr ? d + 32 * u : 0) + quarter * 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (d + 32 * u >= Dr) break;
          float kf[8];
          unpack8<P>(kk[u], kf);
          dots(kf, d + 32 * u);
        }
      }
      weights((rd - br) * 16 + j < n_tok);
#pragma unroll
      for (int u = 0; u < VL; ++u) {
        float vf[8];
        unpack8<P>(vv[u], vf);
        values(vf, u);
      }
      row = next_row;
    }
    store_groups<RH, LPR>(o_s + wave * RH * D, acc, lane);
  }
  __syncthreads();
  for (int x = threadIdx.x; x < RH * D; x += NW * 64) {
    float o = o_s[x];
#pragma unroll 4
    for (int w = 1; w < nact; ++w) o += o_s[w * RH * D + x];
    const float gate = 1.f / (1.f + expf(-proj[(long)t * ld + gate_col + h0 + x / D]));
    out[((long)t * H + h0) * D + x] = P::from_f(o * gate);
  }
}

// ---- prompt attention on the matrix pipe (16-bit storage, D a multiple of 32).
// Workgroup = (16 consecutive positions of one sequence, one key/value group); its four waves take the group's query heads, each wave
// every fourth one in turn.
// Key list of the tile: pooled blocks 0 .. nb(last position), then the tokens from the first position's window start to the last
// position, in steps of 32 keys.  A step is staged ONCE for the four waves: key rows as cached (the A operand of S^T = K Q^T), values
// transposed (the A operand of O^T += V^T P^T); pooled rows, held in fp32, as high and low halves.  The next step's rows are in flight
// while this one is used.  Per step and head:
//   S^T as two 16-key MFMA tiles; P = visible ? sigmoid(S scale + bias) : 0 in fp32, lane (query j, key quad g) holding keys 4g .. 4g+3
//   of both tiles -- which IS the lane's share of the B operand of the value product.
// Scores and weights stay fp32-exact on a bf16 / f16 matrix pipe by splitting the fp32 factor into a high and a low 16-bit
// half (x = hi + lo to 2^-17 in bf16, 2^-22 in fp16): q, the pooled means (held in fp32) and the weights go through two MFMAs instead of one.
// It is bound by the vector work between the products.  With every wave staging its own values, gathering them two bytes at a time and
// testing every key: 38 vector instructions a matrix instruction and 121 us at 2048 positions, 32 + 8 heads of 64, window 512; now 57.
// Token rows that fill their tile (heads of 64, 128, 256) come by LDS-DMA a step ahead, values by transposed reads (seq_rows.h), instead of through registers
// and 2-byte stores: 56.9 us -> 54.1, heads of 128 88.7 -> 82.3, of 256 (16 + 4) 131 -> 112.
// A quarter of that is the sigmoid: with the exponential and the reciprocal as the units give them 45, but its error then grows with the score
// (relative, root mean square in 2^-24: 1.7 within scores of 8 and 6.1 within 30; as below 0.64 and 0.56, a full divide the same).
// 1 / (1 + e^-x): the quotient by one Newton step, which rounds as the divide does
__device__ __forceinline__ float sigmoid_rcp(float x) {
  const float d = 1.f + expf(-x), r = __builtin_amdgcn_rcpf(d), w = fmaf(fmaf(-d, r, 1.f), r, r);
  return d < 1e37f ? w : r;                                // d infinite, or r next to the smallest number: no step
}

template <typename P> __device__ __forceinline__ void split8(const float* v, u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    hi[e] = pack2<P>(v[2 * e], v[2 * e + 1]);
    lo[e] = pack2<P>(v[2 * e] - lo_f<P>(hi[e]), v[2 * e + 1] - hi_f<P>(hi[e]));
  }
}

template <typename P, int NS>
__global__ __launch_bounds__(256) void pwa_attend_mfma_kernel(u16* __restrict__ out, const float* __restrict__ q, UmbPagedKV kv,
                                                              const float* __restrict__ proj, int ld, int gate_col,
                                                              const u16* __restrict__ pos_bias, const int* __restrict__ seq_slot,
                                                              const int* __restrict__ seq_row0, const int* __restrict__ seq_pos0,
                                                              const int* __restrict__ seq_len, int H, int G, int window, int pool,
                                                              float scale) {
  constexpr int D = NS * 32, LD = D + 8, LT = 36, NL = (D + 63) / 64;   // row strides of the two tiles; 8-feature chunks of a row per thread
  extern __shared__ __attribute__((aligned(16))) u16 pwa_lds[];
  u16* k_hi = pwa_lds;                                         // [32][LD]
  u16* v_hi = k_hi + 32 * LD;                              // [D][LT]
  u16* k_lo = v_hi + D * LT;                               // the low halves of pooled rows
  u16* v_lo = k_lo + 32 * LD;
  typedef RowLanes<4 * NS, 4> KeyLanes;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, j = lane & 15, g4 = lane >> 4;
  const KeyLanes key_rows(reinterpret_cast<const u16*>(kv.k), wave, lane), value_rows(reinterpret_cast<const u16*>(kv.v), wave, lane);
  const int b = blockIdx.y, g = blockIdx.z;
  const int n = seq_len[b], q0 = blockIdx.x * 16;
  if (q0 >= n) return;                                     // the whole workgroup
  const int slot = seq_slot[b], row0 = seq_row0[b], pos0 = seq_pos0[b];
  const int nq = n - q0 < 16 ? n - q0 : 16;
  const int i_first = pos0 + q0, i_last = i_first + nq - 1;
  const bool q_ok = j < nq;
  const int i_j = i_first + (q_ok ? j : nq - 1);
  const long qrow = row0 + q0 + (q_ok ? j : nq - 1);
  const int nb_j = i_j - window + 1 >= pool ? (i_j - window + 1) / pool : 0;
  const int nb_first = i_first - window + 1 >= pool ? (i_first - window + 1) / pool : 0;
  const int nb_max = i_last - window + 1 >= pool ? (i_last - window + 1) / pool : 0;
  const int j_lo = i_first - window + 1 > 0 ? i_first - window + 1 : 0, n_tok = i_last - j_lo + 1;
  const int R = H / G;
  const int sm = threadIdx.x & 31, sc = threadIdx.x >> 5;  // staging role: key row sm of the step, 8-feature chunks sc, sc + 8, ..
  for (int r0 = 0; r0 < R; r0 += 4) {                      // a wave without a head still stages and meets the barriers
    const bool active = r0 + wave < R;
    const int h = g * R + (active ? r0 + wave : R - 1);
    u32x4 qhi[NS], qlo[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      float v[8];
      const f32x4 x = *reinterpret_cast<const f32x4*>(q + qrow * H * D + (long)h * D + 32 * s + 8 * g4);
      const f32x4 y = *reinterpret_cast<const f32x4*>(q + qrow * H * D + (long)h * D + 32 * s + 8 * g4 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) { v[e] = x[e]; v[4 + e] = y[e]; }
      split8<P>(v, qhi[s], qlo[s]);
    }
    const float bias = pos_bias ? P::to_f(pos_bias[h]) : 0.f;
    f32x4 o[2 * NS];
#pragma unroll
    for (int dt = 0; dt < 2 * NS; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto put = [&](u16* ks, u16* vt, int ch, u32x4 kk, u32x4 vv) {
      *reinterpret_cast<u32x4*>(ks + sm * LD + 8 * ch) = kk;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vt[(8 * ch + 2 * e) * LT + sm] = (u16)(vv[e] & 0xffffu);
        vt[(8 * ch + 2 * e + 1) * LT + sm] = (u16)(vv[e] >> 16);
      }
    };
    auto key_tile = [&](const u16* ks, int u, int s) { return *reinterpret_cast<const u32x4*>(ks + (16 * u + j) * LD + 32 * s + 8 * g4); };
    auto value_tile = [&](const u16* vt, int dt) {
      const u16* vr = vt + (16 * dt + j) * LT + 4 * g4;
      const u32x2 t0 = *reinterpret_cast<const u32x2*>(vr), t1 = *reinterpret_cast<const u32x2*>(vr + 16);
      return u32x4{t0[0], t0[1], t1[0], t1[1]};
    };
    // whole: every key of the step is seen by every query (rows past the last are not stored); else lane's key 16 u + 4 g4 + rr by `sees`
    auto weights = [&](f32x4 (&s2)[2], bool whole, auto sees, u32x4& hi, u32x4& lo) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = sigmoid_rcp(s2[e >> 2][e & 3] * scale + bias);
      if (!whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = q_ok && sees(16 * (e >> 2) + 4 * g4 + (e & 3)) ? w[e] : 0.f;
      }
      split8<P>(w, hi, lo);
    };

    // ---- pooled blocks: fp32 rows
    f32x4 pk[NL][2], pv[NL][2];
    auto fetch_pooled = [&](int base) {
      const long off = (long)pkv_blk_row(kv, slot, min(base + sm, nb_max - 1), pool, g, G) * D;
#pragma unroll
      for (int u = 0; u < NL; ++u) {
        const int ch = sc + 8 * u;
        if (D % 64 == 0 || ch < D / 8) {
          pk[u][0] = *reinterpret_cast<const f32x4*>(kv.kp + off + 8 * ch);
          pk[u][1] = *reinterpret_cast<const f32x4*>(kv.kp + off + 8 * ch + 4);
          pv[u][0] = *reinterpret_cast<const f32x4*>(kv.vp + off + 8 * ch);
          pv[u][1] = *reinterpret_cast<const f32x4*>(kv.vp + off + 8 * ch + 4);
        }
      }
    };
    if (nb_max > 0) fetch_pooled(0);
    for (int base = 0; base < nb_max; base += 32) {
      __syncthreads();                                     // every wave is done with the previous tile
#pragma unroll
      for (int u = 0; u < NL; ++u) {
        const int ch = sc + 8 * u;
        if (D % 64 == 0 || ch < D / 8) {
          u32x4 kh, kl, vh, vl;
          float t[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = pk[u][e >> 2][e & 3];
          split8<P>(t, kh, kl);
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = pv[u][e >> 2][e & 3];
          split8<P>(t, vh, vl);
          put(k_hi, v_hi, ch, kh, vh);
          put(k_lo, v_lo, ch, kl, vl);
        }
      }
      __syncthreads();
      if (base + 32 < nb_max) fetch_pooled(base + 32);
      if (!active) continue;
      f32x4 s2[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const u32x4 kh = key_tile(k_hi, u, s);
          s2[u] = P::mfma(kh, qlo[s], s2[u]);
          s2[u] = P::mfma(key_tile(k_lo, u, s), qhi[s], s2[u]);
          s2[u] = P::mfma(kh, qhi[s], s2[u]);
        }
      u32x4 phi, plo;
      weights(s2, base + 32 <= nb_first, [&](int k) { return base + k < nb_j; }, phi, plo);
#pragma unroll
      for (int dt = 0; dt < 2 * NS; ++dt) {
        const u32x4 vh = value_tile(v_hi, dt);
        o[dt] = P::mfma(vh, plo, o[dt]);
        o[dt] = P::mfma(value_tile(v_lo, dt), phi, o[dt]);
        o[dt] = P::mfma(vh, phi, o[dt]);
      }
    }

    // ---- tokens
    auto token_step = [&](int base, auto key_of, auto value_of) __attribute__((always_inline)) {
      f32x4 s2[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const u32x4 kh = key_of(u, s);
          s2[u] = P::mfma(kh, qlo[s], s2[u]);
          s2[u] = P::mfma(kh, qhi[s], s2[u]);
        }
      const int jt = j_lo + base;
      u32x4 phi, plo;
      weights(s2, jt + 31 <= i_first && jt > i_last - window, [&](int k) { return jt + k <= i_j && jt + k > i_j - window; }, phi, plo);
#pragma unroll
      for (int dt = 0; dt < 2 * NS; ++dt) {
        const u32x4 vh = value_of(dt);
        o[dt] = P::mfma(vh, plo, o[dt]);
        o[dt] = P::mfma(vh, phi, o[dt]);
      }
    };
    if constexpr (KeyLanes::OK) {                          // by LDS-DMA, a step ahead (seq_rows.h)
      constexpr unsigned HALF = KeyLanes::R::BYTES, BUF = 2 * HALF;
      const unsigned lds0 = (unsigned)(size_t)(lds_char*)pwa_lds;
      unsigned* tab = reinterpret_cast<unsigned*>(pwa_lds + BUF);          // [2][32] behind two buffers of a step's key rows and value rows
      const int steps = (n_tok + 31) / 32;
      auto row_pos = [&](int x) { return j_lo + min(x, n_tok - 1); };
      auto issue = [&](int st) __attribute__((always_inline)) {
        key_rows.issue(tab + (st & 1) * 32, lds0 + (unsigned)(st & 1) * BUF, wave);
        value_rows.issue(tab + (st & 1) * 32, lds0 + (unsigned)(st & 1) * BUF + HALF, wave);
      };
      RowKeys<4 * NS> keys(j, g4);
      RowValues<4 * NS> values(j, g4);
      RowAsked next{};
      __syncthreads();                                     // every wave is done with what stood there
      if (threadIdx.x < 64) tab[threadIdx.x] = pkv_tok_row(kv, slot, row_pos(threadIdx.x), g, G);
      if (threadIdx.x < 32) next.ask(kv, slot, row_pos(64 + threadIdx.x));
      __syncthreads();
      issue(0);
      for (int st = 0; st < steps; ++st) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");        // the step's rows have landed, the step before is read
        __builtin_amdgcn_s_barrier();
        if (threadIdx.x < 32) tab[(st & 1) * 32 + threadIdx.x] = next.row(kv, g, G);
        if (st + 1 < steps) issue(st + 1);
        if (threadIdx.x < 32) next.ask(kv, slot, row_pos(32 * st + 96 + threadIdx.x));
        if (!active) continue;
        keys.at_step(lds0 + (unsigned)(st & 1) * BUF);
        values.at_step(lds0 + (unsigned)(st & 1) * BUF + HALF);
        token_step(32 * st, keys, values);
      }
    } else {
      u32x4 tk[NL], tv[NL];
      auto fetch_tokens = [&](int base) {
        const long off = (long)pkv_tok_row(kv, slot, j_lo + min(base + sm, n_tok - 1), g, G) * D;
#pragma unroll
        for (int u = 0; u < NL; ++u) {
          const int ch = sc + 8 * u;
          if (D % 64 == 0 || ch < D / 8) {
            tk[u] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const u16*>(kv.k) + off + 8 * ch);
            tv[u] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const u16*>(kv.v) + off + 8 * ch);
          }
        }
      };
      fetch_tokens(0);
      for (int base = 0; base < n_tok; base += 32) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NL; ++u) {
          const int ch = sc + 8 * u;
          if (D % 64 == 0 || ch < D / 8) put(k_hi, v_hi, ch, tk[u], tv[u]);
        }
        __syncthreads();
        if (base + 32 < n_tok) fetch_tokens(base + 32);
        if (!active) continue;
        token_step(base, [&](int u, int s) { return key_tile(k_hi, u, s); }, [&](int dt) { return value_tile(v_hi, dt); });
      }
    }
    // lane holds O^T[d = 16 dt + 4 g4 + rr][query j]
    if (q_ok && active) {
      const float gate = 1.f / (1.f + expf(-proj[qrow * ld + gate_col + h]));
#pragma unroll
      for (int dt = 0; dt < 2 * NS; ++dt) {
        u32x2 pk2;
        pk2[0] = pack2<P>(o[dt][0] * gate, o[dt][1] * gate);
        pk2[1] = pack2<P>(o[dt][2] * gate, o[dt][3] * gate);
        *reinterpret_cast<u32x2*>(out + qrow * H * D + (long)h * D + 16 * dt + 4 * g4) = pk2;
      }
    }
  }
}

static inline bool pkv_ok(const UmbPagedKV* kv) {
  return kv && kv->k && kv->v && kv->kp && kv->vp && kv->pages && kv->page >= 1 && kv->max_pages >= 1;
}

static inline bool prep_in_fours(long n, int D) { return n >= 16384 && D <= 128 && D % 2 == 0; }      // from two rounds of waves over the chip on
static int pwa_prep(float* q, const UmbPagedKV* kv, const float* proj, int ld, const int* pos, const int* slot, const float* freq, int T, int H, int G, int D,
                    int rot_dims, float eps, int pool, int dtype, hipStream_t st) {
  if (T < 1 || H < 1 || G < 1 || D < 1 || rot_dims < 0 || rot_dims > D || (rot_dims & 1) || !q || !pkv_ok(kv) || !proj || !pos ||
      !slot || (rot_dims && !freq))
    return UMB_EINVAL;
  const int eb = dtype == UMB_SEQ_F32 ? 4 : 2;
  if (prep_in_fours((long)T * (H + G), D) && (D == 64 || D == 128) && rot_dims % 4 == 0 && (uintptr_t)q % 16 == 0 &&
      ((uintptr_t)kv->k | (uintptr_t)kv->v) % (4 * eb) == 0) {
    const int waves = (H + G + prep_rows(D) - 1) / prep_rows(D);
    const dim3 grid((unsigned)(((long)T * waves + 3) / 4));
    DISPATCH_SEQ_DTYPE(dtype, {
      if (D == 64) hipLaunchKernelGGL((pwa_prep_quads_kernel<P, 64>), grid, dim3(256), 0, st, q, *kv, proj, ld, pos, slot, freq, T, H, G, rot_dims, eps, waves);
      else hipLaunchKernelGGL((pwa_prep_quads_kernel<P, 128>), grid, dim3(256), 0, st, q, *kv, proj, ld, pos, slot, freq, T, H, G, rot_dims, eps, waves);
    })
    UMB_LAUNCH_CHECK();
    return UMB_OK;
  }
  if (prep_in_fours((long)T * (H + G), D)) {
    const int groups = (H + G + 3) / 4;
    DISPATCH_SEQ_DTYPE(dtype, {
      hipLaunchKernelGGL(pwa_prep_four_kernel<P>, dim3((unsigned)(((long)T * groups + 3) / 4)), dim3(256), 0, st, q, *kv, proj, ld, pos, slot,
                         freq, T, H, G, D, rot_dims, eps, groups);
    })
    UMB_LAUNCH_CHECK();
    return UMB_OK;
  }
  const long n = (long)T * (H + G + (pool > 0 ? G : 0));
  DISPATCH_SEQ_DTYPE(dtype, {
    hipLaunchKernelGGL(pwa_prep_kernel<P>, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, q, *kv, proj, ld, pos, slot, freq, T, H,
                       G, D, rot_dims, eps, pool);
  })
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
extern "C" int umb_pwa_prep(float* q, const UmbPagedKV* kv, const float* proj, int ld, const int* pos, const int* slot,
                            const float* freq, int T, int H, int G, int D, int rot_dims, float eps, int dtype, hipStream_t st) {
  return pwa_prep(q, kv, proj, ld, pos, slot, freq, T, H, G, D, rot_dims, eps, 0, dtype, st);
}
extern "C" int umb_pwa_prep_step(float* q, const UmbPagedKV* kv, const float* proj, int ld, const int* pos, const int* slot, const float* freq,
                                 const int* seq_slot, const int* seq_pos0, const int* seq_len, int T, int H, int G, int D, int rot_dims, int pool,
                                 float eps, int dtype, hipStream_t st) {
  if (pool < 1 || !seq_slot || !seq_pos0 || !seq_len || !kv || !kv->kp || !kv->vp) return UMB_EINVAL;
  const int rc = pwa_prep(q, kv, proj, ld, pos, slot, freq, T, H, G, D, rot_dims, eps, pool, dtype, st);
  return rc == UMB_OK && prep_in_fours((long)T * (H + G), D) ? umb_pwa_pool(kv, seq_slot, seq_pos0, seq_len, T, 1, G, D, pool, dtype, st) : rc;
}
extern "C" int umb_pwa_pool(const UmbPagedKV* kv, const int* seq_slot, const int* seq_pos0, const int* seq_len, int B, int max_len,
                            int G, int D, int pool, int dtype, hipStream_t st) {
  if (B < 1 || max_len < 1 || G < 1 || D < 1 || pool < 1 || !pkv_ok(kv) || !seq_slot || !seq_pos0 || !seq_len) return UMB_EINVAL;
  const int nb = max_len / pool + 1;             // at most this many blocks end inside max_len consecutive positions
  DISPATCH_SEQ_DTYPE(dtype, {
    hipLaunchKernelGGL(pwa_pool_kernel<P>, dim3(nb, B, G), dim3(D > 192 ? 256 : (D + 63) / 64 * 64), 0, st, *kv, seq_slot, seq_pos0, seq_len, G, D, pool);
  })
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// single tokens (seq_decode.h); prep: prepared here, of one token a sequence
static int pwa_decode(void* out, const float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col, const void* pos_bias, const int* pos,
                    const int* slot, int T, int H, int G, int D, int window, int pool, float scale, int dtype, const PwaPrep* prep, hipStream_t st) {
  const int R = H / G;
  // 16 waves per item as long as every item gets a compute unit of its own, 8 while two share one, 4 beyond (us with 8 / 4 waves, 32 + 8 heads of
  // 64: 1024 items behind 30 / 200 keys 12.7 / 7.8, 24.9 / 20.1, 768 behind 200 19.1 / 12.9; 512 items of 128 behind 500 25.4 / 30.0)
  const int rh = R % 4 == 0 && (long)T * H > 128 ? 4 : (R % 2 == 0 ? 2 : 1);       // few rows in all: two a workgroup, as in seq_battn.hip
  const long items = (long)T * (H / rh);
  const int nw = items <= 256 ? 16 : (items <= 512 ? 8 : 4);
  const size_t lds = (size_t)nw * rh * D * sizeof(float);
#define PWD_GO_AS(RH, LPR, NW, PREP, ARG)                                                                                       \
  do {                                                                                                                          \
  if (ensure_dynamic_lds<pwa_decode_kernel<P, RH, LPR, NW, PREP>>(lds) != UMB_OK) return UMB_EHIP;                            \
  hipLaunchKernelGGL((pwa_decode_kernel<P, RH, LPR, NW, PREP>), dim3(T, H / rh), dim3(NW * 64), lds, st, (u16*)out, q, *kv, proj, ld, \
                     gate_col, (const u16*)pos_bias, pos, slot, H, G, D, window, pool, scale, ARG);                           \
  } while (0)
#define PWD_GO(RH, LPR, NW) do { if (prep) PWD_GO_AS(RH, LPR, NW, true, *prep); else PWD_GO_AS(RH, LPR, NW, false, PwaPrep{}); } while (0)
#define PWD_NW(RH, LPR) do { if (nw == 16) PWD_GO(RH, LPR, 16); else if (nw == 8) PWD_GO(RH, LPR, 8); else PWD_GO(RH, LPR, 4); } while (0)
#define PWD_RH(LPR) do { if (rh == 4) PWD_NW(4, LPR); else if (rh == 2) PWD_NW(2, LPR); else PWD_NW(1, LPR); } while (0)
#define PWD_D() do { if (D == 64) PWD_RH(8); else if (D == 128) PWD_RH(16); else PWD_RH(32); } while (0)
  if (dtype == UMB_SEQ_BF16) { using P = BF16; PWD_D(); }
  else { using P = F16; PWD_D(); }
#undef PWD_D
#undef PWD_RH
#undef PWD_NW
#undef PWD_GO
#undef PWD_GO_AS
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
extern "C" int umb_pwa_attend(void* out, const float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col,
                              const void* pos_bias, const int* pos, const int* slot, int T, int H, int G, int D, int window,
                              int pool, float scale, int dtype, hipStream_t st) {
  if (T < 1 || H < 1 || G < 1 || H % G || D < 1 || D > 64 * PWA_MAXC || window < 1 || pool < 1 || !out || !q || !pkv_ok(kv) ||
      !proj || !pos || !slot)
    return UMB_EINVAL;
  if (decode_rows_ok(D, D, dtype, kv))
    return pwa_decode(out, q, kv, proj, ld, gate_col, pos_bias, pos, slot, T, H, G, D, window, pool, scale, dtype, nullptr, st);
  const int R = H / G;
  const int rh = R % 8 == 0 ? 8 : (R % 4 == 0 ? 4 : (R % 2 == 0 ? 2 : 1));     // heads of one group per workgroup
  const int Dp = (D + 3) & ~3;
  const dim3 grid(T, H / rh);
  // few workgroups (decoding): sixteen waves share a query's keys, so a step's latency is one or two rounds; many (prompts):
  // four, the chip is full anyway.  The choice changes the order in which a query's partial sums are added, nothing else.
  int nw = (long)T * (H / rh) < 1024 ? 16 : 4;
  if (nw == 16 && ((size_t)16 * rh * Dp + 16 * (rh * 64 + 128)) * sizeof(float) > 96 * 1024) nw = 4;     // LDS of one CU
  const size_t lds = ((size_t)nw * rh * Dp + nw * (rh * 64 + 128)) * sizeof(float);
#define PWA_LAUNCH(RH, NC, NW)                                                                                            \
  do {                                                                                                                    \
    if (ensure_dynamic_lds<pwa_attend_kernel<P, RH, NC, NW>>(lds) != UMB_OK) return UMB_EHIP;                             \
    hipLaunchKernelGGL((pwa_attend_kernel<P, RH, NC, NW>), grid, dim3(NW * 64), lds, st, (E*)out, q, *kv, proj, ld,       \
                       gate_col, (const E*)pos_bias, pos, slot, T, H, G, D, window, pool, scale);                         \
  } while (0)
#define PWA_NC(RH, NW)                                                                                                    \
  if (D <= 64) PWA_LAUNCH(RH, 1, NW); else if (D <= 128) PWA_LAUNCH(RH, 2, NW); else PWA_LAUNCH(RH, 4, NW)
#define PWA_CASE(RH)                                                                                                       \
  case RH:                                                                                                                 \
    if (nw == 16) { PWA_NC(RH, 16); } else { PWA_NC(RH, 4); }                                                              \
    break;
  DISPATCH_SEQ_DTYPE(dtype, {
    typedef typename El<P>::type E;
    switch (rh) { PWA_CASE(8) PWA_CASE(4) PWA_CASE(2) default: PWA_CASE(1) }
  })
#undef PWA_CASE
#undef PWA_NC
#undef PWA_LAUNCH
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_pwa_step(void* out, float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col, const void* pos_bias, const int* pos,
                            const int* slot, const float* freq, const int* seq_slot, const int* seq_pos0, const int* seq_len, int T, int H, int G, int D,
                            int rot_dims, int window, int pool, float scale, float eps, int dtype, hipStream_t st) {
  if (T < 1 || H < 1 || G < 1 || H % G || D < 1 || D > 64 * PWA_MAXC || window < 1 || pool < 1 || rot_dims < 0 || rot_dims > D || (rot_dims & 1) || !out || !q ||
      !pkv_ok(kv) || !proj || !pos || !slot || (rot_dims && !freq) || !seq_slot || !seq_pos0 || !seq_len)
    return UMB_EINVAL;
  if (decode_rows_ok(D, D, dtype, kv)) {
    const PwaPrep prep{freq, rot_dims, eps};
    return pwa_decode(out, nullptr, kv, proj, ld, gate_col, pos_bias, pos, slot, T, H, G, D, window, pool, scale, dtype, &prep, st);
  }
  const int rc = umb_pwa_prep_step(q, kv, proj, ld, pos, slot, freq, seq_slot, seq_pos0, seq_len, T, H, G, D, rot_dims, pool, eps, dtype, st);
  return rc != UMB_OK ? rc : umb_pwa_attend(out, q, kv, proj, ld, gate_col, pos_bias, pos, slot, T, H, G, D, window, pool, scale, dtype, st);
}

extern "C" int umb_pwa_attend_tiled(void* out, const float* q, const UmbPagedKV* kv, const float* proj, int ld, int gate_col,
                                    const void* pos_bias, const int* seq_slot, const int* seq_row0, const int* seq_pos0,
                                    const int* seq_len, int B, int max_len, int H, int G, int D, int window, int pool, float scale,
                                    int dtype, hipStream_t st) {
  if (B < 1 || max_len < 1 || H < 1 || G < 1 || H % G || D < 32 || D > 256 || D % 32 || window < 1 || pool < 1 || !out || !q ||
      !pkv_ok(kv) || !proj || !seq_slot || !seq_row0 || !seq_pos0 || !seq_len || dtype == UMB_SEQ_F32)
    return UMB_EINVAL;
  const dim3 grid((max_len + 15) / 16, B, G);
  const size_t lds = 2 * ((size_t)32 * (D + 8) + (size_t)D * 36) * sizeof(u16);      // pooled tiles; two steps of token rows and their table are less
#define PWA_MFMA_CASE(NS)                                                                                                  \
  case NS:                                                                                                                 \
    if (ensure_dynamic_lds<pwa_attend_mfma_kernel<P, NS>>(lds) != UMB_OK) return UMB_EHIP;                                 \
    hipLaunchKernelGGL((pwa_attend_mfma_kernel<P, NS>), grid, dim3(256), lds, st, (u16*)out, q, *kv, proj, ld, gate_col,   \
                       (const u16*)pos_bias, seq_slot, seq_row0, seq_pos0, seq_len, H, G, window, pool, scale);            \
    break;
  if (dtype == UMB_SEQ_BF16) {
    using P = BF16;
    switch (D / 32) { PWA_MFMA_CASE(1) PWA_MFMA_CASE(2) PWA_MFMA_CASE(3) PWA_MFMA_CASE(4) PWA_MFMA_CASE(5) PWA_MFMA_CASE(6)
                      PWA_MFMA_CASE(7) PWA_MFMA_CASE(8) default: return UMB_EINVAL; }
  } else if (dtype == UMB_SEQ_F16) {
    using P = F16;
    switch (D / 32) { PWA_MFMA_CASE(1) PWA_MFMA_CASE(2) PWA_MFMA_CASE(3) PWA_MFMA_CASE(4) PWA_MFMA_CASE(5) PWA_MFMA_CASE(6)
                      PWA_MFMA_CASE(7) PWA_MFMA_CASE(8) default: return UMB_EINVAL; }
  } else {
    return UMB_EINVAL;
  }
#undef PWA_MFMA_CASE
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
