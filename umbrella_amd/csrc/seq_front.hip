// A few rows' seam (seq_norm.hip, seq_hyper.hip) inside the product that reads it: out = product(h), h the rows that the seam would have left in
// memory, and the new residual rows beside it.
//
// A seam of one row is latency alone: a launch, one trip to memory, two sums, the rows written back and read again by the product behind it, 4.5 us for
// 100 KB.  Every workgroup of the product can form the rows itself in less: its weights are asked for first, and the rows' operands, some 50 KB from
// the caches, arrive beside them.  Four waves fetch weights and multiply, as in seq_linear.hip; four others form the rows in LDS and end (their loads
// are waited for on a counter of their own: in the same wave a wait for the rows would be one for the weights in front of them).  Of a product's
// workgroups each reads all rows, so this is for rows of a few thousand elements together: front_form.
// The arithmetic is the seams' and the products', sum for sum: a step's results are the same bits whichever way its seams run, and do not depend on
// how many of these few rows it has.  The residual is read by every workgroup and therefore not written in place: x_out is another buffer.
#include "seq_linear.h"

constexpr int FRONT_MAX = 16;      // sets of 64 quads in all rows
// SETS: those that a wave of four forms.  Its registers hold a set's every operand; the slabs of a split output only where they fit beside them.
template <typename P, int KIND, int SETS> constexpr bool front_slabs() { return SETS <= 2 || (KIND != UMB_FRONT_PAIR && sizeof(typename El<P>::type) == 2); }

// four weights as they are stored
template <typename P> struct Quad {
  u32x2 v;
  __device__ __forceinline__ void load(const void* p, int i) { v = *reinterpret_cast<const u32x2*>(reinterpret_cast<const u16*>(p) + i); }
  __device__ __forceinline__ f32x4 get() const { return f32x4{lo_f<P>(v[0]), hi_f<P>(v[0]), lo_f<P>(v[1]), hi_f<P>(v[1])}; }
};
template <> struct Quad<F32> {
  f32x4 v;
  __device__ __forceinline__ void load(const void* p, int i) { v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p) + i); }
  __device__ __forceinline__ f32x4 get() const { return v; }
};

// Sums over the wave of up to four values: the lanes' row r (16 of them) ends up with value r's, the pairs that wave_sum adds in the order that it adds
// them.  Four sums in 10 instructions: what is executed once a launch costs its fetch (a code of 17 KB, four sums and quotients one by one, took 5 us).
template <int CTRL> __device__ __forceinline__ float dpp_add(float v) {
  return v + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), CTRL, 0xf, 0xf, false));
}
// x[l] of a row of 16 lanes + x[l ^ 8], then ^ 4, 2, 1 (rotations: behind the first the row repeats itself)
__device__ __forceinline__ float row16_sum(float v) { return dpp_add<0x121>(dpp_add<0x122>(dpp_add<0x124>(dpp_add<0x128>(v)))); }
template <int SETS> __device__ __forceinline__ float sets_sum(const float (&v)[SETS]) {
  static_assert(SETS == 2 || SETS == 4);
  auto half = [](float a, float b) {       // lanes 0 - 31: a + its other half, 32 - 63: b's
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
  };
  const float p = half(v[0], SETS == 4 ? v[SETS / 2] : v[1]), q = SETS == 4 ? half(v[1], v[SETS - 1]) : p;      // (values 0 and 2, 1 and 3)
  const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(p), __float_as_uint(q), false, false);
  return row16_sum(__uint_as_float(t[0]) + __uint_as_float(t[1]));
}
// lane row that holds value i
template <int SETS> __device__ __forceinline__ constexpr int set_row(int i) { return SETS == 4 ? i : 2 * i; }
// barriers that the rows take: behind the requests, the sums, the rows themselves
template <int KIND> constexpr int front_barriers() { return 1 + (KIND == UMB_FRONT_SEAM ? 3 : KIND == UMB_FRONT_PAIR ? 4 : 2); }

// wave u of four: sets u, u + 4, ... of the rows' quads (64 consecutive quads of a (row, group) each) to LDS, rows hs bytes apart; the last barrier is the
// caller's.  behind(): what is to follow the requests of the rows -- memory answers in order, and a unit's weights in front of them were 4 us of waiting.
template <typename P, int KIND, int SETS, typename Behind>
__device__ __forceinline__ void front_rows(const UmbSeqFront& f, int T, unsigned char* h, unsigned hs, float (*sums)[FRONT_MAX + 16], int u, int lane,
                                           float* __restrict__ x_out, Behind behind) {
  typedef typename El<P>::type E;
  const int W = f.W, groups = KIND == UMB_FRONT_SEAM || KIND == UMB_FRONT_EMBED ? f.groups : 1, gs = W / groups, nq = gs / 4, spg = (nq + 63) / 64;
  const int nsets = T * groups * spg, slab = T * W;
  const float len = (float)gs, eps = f.eps;
  constexpr bool LATE = KIND == UMB_FRONT_PAIR && SETS > 2;       // two of a pair's weights behind the first sums: the registers of long rows
  int col[SETS], row[SETS], first[SETS];
  bool in[SETS];
  f32x4 y[SETS], y2[SETS], x[SETS];
  Quad<P> wp[SETS], wn[SETS], w1[SETS], w2[SETS];      // as stored until they are used
#pragma unroll
  for (int i = 0; i < SETS; ++i) {
    const int s = u + 4 * i, sc = min(s, nsets - 1), unit = __builtin_amdgcn_readfirstlane(sc / spg), q = (sc - unit * spg) * 64 + lane;      // unit: (row, group)
    row[i] = __builtin_amdgcn_readfirstlane(unit / groups);
    in[i] = s < nsets && q < nq;
    first[i] = unit * spg;
    col[i] = (unit - row[i] * groups) * gs + min(q, nq - 1) * 4;
  }
  auto at = [&](const float* p, int i) { return reinterpret_cast<const f32x4*>(p + (long)(row[i] * W) + col[i]); };
#pragma unroll
  for (int i = 0; i < SETS; ++i) {
    if constexpr (KIND == UMB_FRONT_EMBED) {
      const int tok = min(max(f.tokens[row[i]], 0), f.V - 1);
      x[i] = ld4<P>(reinterpret_cast<const E*>(f.embed) + (long)tok * W + col[i]) * f.scale;
    } else {
      y[i] = *at(f.y, i);
      x[i] = *at(f.x, i);
    }
    if constexpr (!LATE) {
      wn[i].load(f.w_next, col[i]);
      if constexpr (KIND == UMB_FRONT_SEAM || KIND == UMB_FRONT_PAIR) wp[i].load(f.w_post, col[i]);
    }
    if constexpr (KIND == UMB_FRONT_PAIR) {
      y2[i] = *at(f.y2, i);
      w1[i].load(f.w1, col[i]);
      w2[i].load(f.w2, col[i]);
    }
  }
  f32x4 part[2][3][SETS];
  auto ask = [&](f32x4 (&v)[3][SETS], const float* src, int parts) __attribute__((always_inline)) {
    if constexpr (front_slabs<P, KIND, SETS>()) {
#pragma unroll
      for (int p = 0; p < 3; ++p)
        if (parts > p + 1)
#pragma unroll
          for (int i = 0; i < SETS; ++i) v[p][i] = *at(src + (p + 1) * slab, i);
    }
  };
  auto add = [&](f32x4 (&to)[SETS], const f32x4 (&v)[3][SETS], int parts) __attribute__((always_inline)) {
    if constexpr (front_slabs<P, KIND, SETS>()) {
#pragma unroll
      for (int p = 0; p < 3; ++p)
        if (parts > p + 1)
#pragma unroll
          for (int i = 0; i < SETS; ++i) to[i] += v[p][i];
    }
  };
  if constexpr (KIND != UMB_FRONT_EMBED) ask(part[0], f.y, f.parts);
  if constexpr (KIND == UMB_FRONT_PAIR) ask(part[1], f.y2, f.parts2);
  behind();
  if constexpr (KIND != UMB_FRONT_EMBED) add(y, part[0], f.parts);
  if constexpr (KIND == UMB_FRONT_PAIR) add(y2, part[1], f.parts2);

  const int mine = lane >> 4, lead = lane & 15;                   // this lane's row and place in it
  auto squares = [&](const f32x4 (&v)[SETS], int which) __attribute__((always_inline)) {
    float s[SETS];
#pragma unroll
    for (int i = 0; i < SETS; ++i) s[i] = in[i] ? sq4(v[i]) : 0.f;
    const float t = sets_sum(s);
    if (lead == 0) sums[which][SETS == 4 ? u + 4 * mine : (mine & 1) ? FRONT_MAX + mine : u + 2 * mine] = t;      // (sets that are none: never read)
  };
  // num / sqrt(mean + eps) of every set's (row, group), the parts of its sum in pairs as row_sum adds them (those it does not have are zeros there)
  auto factors = [&](float (&g)[SETS], float num, int which) __attribute__((always_inline)) {
    int from = first[0];
#pragma unroll
    for (int i = 1; i < SETS; ++i) from = mine >= set_row<SETS>(i) ? first[i] : from;
    const float t = row16_sum(lead < spg ? sums[which][from + lead] : 0.f), q = num / sqrtf(t / len + eps);
#pragma unroll
    for (int i = 0; i < SETS; ++i) g[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(q), 16 * set_row<SETS>(i)));
  };
  float g[SETS], gb[SETS];
  auto leave = [&](int i) __attribute__((always_inline)) {        // the new residual
    if (x_out && in[i]) *reinterpret_cast<f32x4*>(x_out + (long)(row[i] * W) + col[i]) = x[i];
  };
  constexpr int LAST = KIND == UMB_FRONT_SEAM ? 1 : KIND == UMB_FRONT_PAIR ? 3 : 0;      // the sum that the next norm divides by
  if constexpr (KIND == UMB_FRONT_SEAM) {
    squares(y, 0);
    __syncthreads();
    factors(g, 1.f, 0);
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
      x[i] = x[i] + y[i] * g[i] * wp[i].get();
      leave(i);
    }
  } else if constexpr (KIND == UMB_FRONT_PAIR) {
    squares(y, 0);
    squares(y2, 1);
    if constexpr (LATE) {
#pragma unroll
      for (int i = 0; i < SETS; ++i) {
        wn[i].load(f.w_next, col[i]);
        wp[i].load(f.w_post, col[i]);
      }
    }
    __syncthreads();
    factors(g, f.coef, 0);
    factors(gb, f.coef, 1);
#pragma unroll
    for (int i = 0; i < SETS; ++i) y[i] = pair_sum<1>(y[i], g[i], w1[i].get(), y2[i], gb[i], w2[i].get());
    squares(y, 2);
    __syncthreads();
    factors(g, 1.f, 2);
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
      x[i] = x[i] + y[i] * g[i] * wp[i].get();
      leave(i);
    }
  } else {
    const float in0 = f.in ? f.in[0] : 1.f;
    const float mx = KIND == UMB_FRONT_STREAM && f.mix ? f.mix[0] : 1.f, ot = KIND == UMB_FRONT_STREAM && f.out ? f.out[0] : 1.f;
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
      if constexpr (KIND == UMB_FRONT_STREAM) x[i] = stream_write<1>(mx, x[i], ot, f.m, y[i]);
      leave(i);
      x[i] = in0 * x[i];
    }
  }
  squares(x, LAST);
  __syncthreads();
  factors(g, 1.f, LAST);
#pragma unroll
  for (int i = 0; i < SETS; ++i) {
    f32x4 v;
    if constexpr (KIND == UMB_FRONT_SEAM || KIND == UMB_FRONT_PAIR) v = x[i] * g[i] * wn[i].get();
    else v = x[i] * g[i] * (f.offset + wn[i].get());
    if (in[i]) st4<P>(reinterpret_cast<E*>(h + row[i] * hs) + col[i], v);
  }
}

// one finished output (l / r as in seq_linear.hip: n = 4 (l / 16) + r, token l % 16)
template <typename P, bool DUAL>
__device__ __forceinline__ void front_store(void* out, long o, float s, float s2, int epi, float limit, float alpha) {
  typedef typename El<P>::type E;
  if constexpr (DUAL) stf<P>(reinterpret_cast<E*>(out) + o, glu_pair(epi, s, s2, limit, alpha));
  else if (epi == EPI_DT) stf<P>(reinterpret_cast<E*>(out) + o, s);
  else if (epi == EPI_RELU2) {
    const float rl = fmaxf(s, 0.f);
    stf<P>(reinterpret_cast<E*>(out) + o, rl * rl);
  } else if (epi == EPI_CAP) reinterpret_cast<float*>(out)[o] = limit * tanhf(s / limit);
  else reinterpret_cast<float*>(out)[o] = s;
}

// ---- K in whole 512-byte pieces: seq_linear_stream_kernel of one token tile, its tokens' rows standing in LDS
template <bool DUAL, int SLOTS> struct FrontRing {
  static constexpr int AP = DUAL ? 16 : 8, R = SLOTS;
  static constexpr unsigned PIECE = 1040u, SLOT = AP * PIECE;
};
template <typename P, bool DUAL, int KIND, int SETS, int SLOTS, bool RUN>
__global__ __launch_bounds__(512, 4) void front_stream_kernel(void* __restrict__ out, const typename El<P>::type* __restrict__ w,
                                                              const typename El<P>::type* __restrict__ bias, int T, int N, int K, int epi, float limit,
                                                              float alpha, int step, int turn, float* __restrict__ x_out, UmbSeqFront f) {
  typedef typename El<P>::type E;
  typedef FrontRing<DUAL, SLOTS> S;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float sums[4][FRONT_MAX + 16];
  constexpr int EB = sizeof(E), STEPS = 512 / (32 * EB), AT = DUAL ? 2 : 1, PW = S::AP / 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned hs = (unsigned)K * EB + 64u;
  if (wave >= 4) {
    front_rows<P, KIND, SETS>(f, T, smem + S::R * S::SLOT, hs, sums, wave - 4, lane, blockIdx.x == 0 ? x_out : nullptr,
                              [] { __syncthreads(); });
    __syncthreads();
    return;
  }
  const int j = lane & 15, g = lane >> 4;
  const unsigned lds0 = (unsigned)(size_t)(lds_char*)smem, hrow = lds0 + S::R * S::SLOT + (unsigned)min(j, T - 1) * hs;
  unsigned voff[PW];
  auto rows_of_block = [&](int n0) {
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int odd = lane >> 5, c = (lane & 31) ^ (odd * 8), r = 2 * (wave + 4 * i) + odd;
      const int n = DUAL && r >= 16 ? N + min(n0 + r - 16, N - 1) : min(n0 + r, N - 1);
      voff[i] = (unsigned)(n - n0) * (unsigned)K * EB + c * 16u;
    }
  };
  const char* wb = reinterpret_cast<const char*>(w);
  const int nc = K * EB / 512, nb = (N + 15) / 16;
  int fb = blockIdx.x, left = nc, col = first_chunk(fb * 16, nc, turn);
  const char* fw = wb + (long)fb * 16 * K * EB;
  rows_of_block(fb * 16);
  auto issue = [&](int slot) {
    const long at = (long)col * 512;
    col = col + 1 == nc ? 0 : col + 1;
    --left;
#pragma unroll
    for (int i = 0; i < PW; ++i) tile_dma_once(voff[i], fw + at, lds0 + (unsigned)slot * S::SLOT + (unsigned)(wave + 4 * i) * S::PIECE);
  };
  __builtin_amdgcn_s_barrier();                             // the rows are asked for
#pragma unroll
  for (int c = 0; c < S::R - 1; ++c) issue(c);
#pragma unroll
  for (int i = 1; i < front_barriers<KIND>(); ++i) __builtin_amdgcn_s_barrier();
  const unsigned wrow = (unsigned)(j >> 1) * S::PIECE + (unsigned)(j & 1) * 512u, swz = (unsigned)(j & 1) * 8u;
  f32x4 acc[AT];
  int slot = 0;
  for (int block = blockIdx.x; block < nb; block += step) {
    const int n0 = block * 16;
#pragma unroll
    for (int i = 0; i < AT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    unsigned base = lds0;
    int at = first_chunk(n0, nc, turn);                     // the chunk that is multiplied
    for (int c = 0; c < nc; ++c) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((S::R - 2) * PW) : "memory");
      __builtin_amdgcn_s_barrier();
      if (RUN && __builtin_expect(left == 0 && fb + step < nb, 0)) {
        fb += step;
        left = nc;
        col = first_chunk(fb * 16, nc, turn);
        fw = wb + (long)fb * 16 * K * EB;
        rows_of_block(fb * 16);
      }
      issue(slot == 0 ? S::R - 1 : slot - 1);
      base = lds0 + (unsigned)slot * S::SLOT;
      const unsigned hb = hrow + (unsigned)at * 512u;
      at = at + 1 == nc ? 0 : at + 1;
#pragma unroll
      for (int v = 0; v < STEPS / 4; ++v) {
        const int s = wave + 4 * v;
        const auto w16 = [&](int i, int cc) { return *reinterpret_cast<const lds_u32x4*>((size_t)(base + (unsigned)(8 * i) * S::PIECE + wrow + (((unsigned)cc) ^ swz) * 16u)); };
        const auto h16 = [&](int cc) { return *reinterpret_cast<const lds_u32x4*>((size_t)(hb + (unsigned)cc * 16u)); };
        Frag8<P> a[AT], b;
        if constexpr (EB == 2) {
#pragma unroll
          for (int i = 0; i < AT; ++i) a[i].v = w16(i, s * 4 + g);
          b.v = h16(s * 4 + g);
        } else {
#pragma unroll
          for (int i = 0; i < AT; ++i) {
            a[i].lo = __builtin_bit_cast(f32x4, w16(i, s * 8 + 2 * g));
            a[i].hi = __builtin_bit_cast(f32x4, w16(i, s * 8 + 2 * g + 1));
          }
          b.lo = __builtin_bit_cast(f32x4, h16(s * 8 + 2 * g));
          b.hi = __builtin_bit_cast(f32x4, h16(s * 8 + 2 * g + 1));
        }
#pragma unroll
        for (int i = 0; i < AT; ++i) acc[i] = mma8<P>(a[i], b, acc[i]);
      }
      slot = slot + 1 == S::R ? 0 : slot + 1;
    }
    if (!RUN || block + step >= nb) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < AT; ++i) *reinterpret_cast<lds_f32x4*>((size_t)(base + ((wave * AT + i) * 256 + lane * 4) * 4u)) = acc[i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const int l = threadIdx.x >> 2, r = threadIdx.x & 3, n = n0 + 4 * (l >> 4) + r, t = l & 15;
    if (n < N && t < T) {
      auto total = [&](int i) {
        const auto part = [&](int ww) { return *reinterpret_cast<const lds_f32*>((size_t)(base + ((ww * AT + i) * 256 + threadIdx.x) * 4u)); };
        float s = part(0);
#pragma unroll
        for (int ww = 1; ww < 4; ++ww) s += part(ww);
        return s;
      };
      const float s = total(0) + (bias ? ldf<P>(bias + n) : 0.f);
      float s2 = 0.f;
      if constexpr (DUAL) s2 = total(1) + (bias ? ldf<P>(bias + N + n) : 0.f);
      front_store<P, DUAL>(out, (long)t * N + n, s, s2, epi, limit, alpha);
    }
    if (!RUN) break;
  }
}

// ---- any other K in whole 8-groups up to 128 UN: seq_linear_kernel of one tile, all its weights asked for in front of the rows
template <typename P, bool DUAL, int KIND, int SETS, int UN>
__global__ __launch_bounds__(256) void front_linear_kernel(void* __restrict__ out, const typename El<P>::type* __restrict__ w,
                                                           const typename El<P>::type* __restrict__ bias, int T, int N, int K, int epi, float limit,
                                                           float alpha, float* __restrict__ x_out, UmbSeqFront f) {
  typedef typename El<P>::type E;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float sums[4][FRONT_MAX + 16];
  __shared__ float red[DUAL ? 2 : 1][4][256];
  constexpr int EB = sizeof(E);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const unsigned hs = (unsigned)K * EB + 64u;
  const E* wrow = w + (long)min((int)blockIdx.x * 16 + j, N - 1) * K;
  const int l = threadIdx.x >> 2, r = threadIdx.x & 3, n = blockIdx.x * 16 + 4 * (l >> 4) + r;
  Frag8<P> a[UN], a2[UN];
  float bv = 0.f, bv2 = 0.f;
  front_rows<P, KIND, SETS>(f, T, smem, hs, sums, wave, lane, blockIdx.x == 0 ? x_out : nullptr, [&] {
#pragma unroll
    for (int s = 0; s < UN; ++s) {
      const int k = wave * 32 + s * 128 + g * 8;
      a[s] = load8<P, true>(wrow, k, K);
      if constexpr (DUAL) a2[s] = load8<P, true>(wrow + (long)N * K, k, K);
    }
    if (bias) {
      bv = ldf<P>(bias + min(n, N - 1));
      if constexpr (DUAL) bv2 = ldf<P>(bias + N + min(n, N - 1));
    }
  });
  __syncthreads();
  const E* hrow = reinterpret_cast<const E*>(smem + min(j, T - 1) * hs);
  f32x4 acc{0.f, 0.f, 0.f, 0.f}, acc2{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < UN; ++s) {
    const Frag8<P> b = load8<P, true>(hrow, wave * 32 + s * 128 + g * 8, K);
    acc = mma8<P>(a[s], b, acc);
    if constexpr (DUAL) acc2 = mma8<P>(a2[s], b, acc2);
  }
  *reinterpret_cast<f32x4*>(&red[0][wave][lane * 4]) = acc;
  if constexpr (DUAL) *reinterpret_cast<f32x4*>(&red[1][wave][lane * 4]) = acc2;
  __syncthreads();
  const int t = l & 15;
  if (n >= N || t >= T) return;
  float s = red[0][0][threadIdx.x], s2 = 0.f;
#pragma unroll
  for (int ww = 1; ww < 4; ++ww) s += red[0][ww][threadIdx.x];
  s += bv;
  if constexpr (DUAL) {
    s2 = red[1][0][threadIdx.x];
#pragma unroll
    for (int ww = 1; ww < 4; ++ww) s2 += red[1][ww][threadIdx.x];
    s2 += bv2;
  }
  front_store<P, DUAL>(out, (long)t * N + n, s, s2, epi, limit, alpha);
}

// 0: not covered; 1: K in whole chunks, where the streaming kernel would take the product; 2: the one-tile kernel
static int front_form(const UmbSeqFront* f, const void* w, int T, int N, int epi, int dtype) {
  if (!f || T < 1 || T > 16 || N < 1 || f->W < 4 || f->kind < 0 || f->kind > UMB_FRONT_EMBED || !w || !f->w_next || !(epi_plain(epi) || epi == EPI_CLAMP_GLU || epi == EPI_CAP))
    return 0;
  if (epi_dual(epi)) {
    if (N & 1) return 0;
    N >>= 1;
  }
  const bool embed = f->kind == UMB_FRONT_EMBED, grouped = f->kind == UMB_FRONT_SEAM || embed;
  const int K = f->W, groups = grouped ? f->groups : 1, eb = (int)seq_elem_bytes(dtype);
  if (groups < 1 || K % groups || (uintptr_t)w % 16) return 0;
  if (!quads_ok(K, groups, embed ? f->embed : f->x, f->y, f->y2, f->w_next, f->w_post, f->w1, f->w2)) return 0;
  if (embed ? !f->embed || !f->tokens || f->V < 1 : !f->x || !f->y || f->parts < 1 || f->parts > PARTS_MAX) return 0;
  if (f->kind == UMB_FRONT_SEAM && !f->w_post) return 0;
  if (f->kind == UMB_FRONT_PAIR && (!f->y2 || !f->w_post || !f->w1 || !f->w2 || f->parts2 < 1 || f->parts2 > PARTS_MAX)) return 0;
  const int gs = K / groups;
  const long sets = (long)T * groups * ((gs + 255) / 256);
  if (gs > 4096 || sets > FRONT_MAX || K % 8) return 0;
  // (front_slabs; a pair of fp32 weights does not fit the registers either way)
  if (sets > 8 && ((f->kind == UMB_FRONT_PAIR && (eb == 4 || f->parts > 1 || f->parts2 > 1)) || (!embed && eb == 4 && f->parts > 1))) return 0;
  // Where it pays: the rows are reading in every workgroup, in place of the seam's launch.  Up to eight sets, in however many rows, that is less wherever the
  // streaming kernel runs; more sets are where they are one row's, or workgroups few.  us, the seam and the product / this, bf16: one row of 4096, N 4096 10.9 / 10.1,
  // 6144 13.5 / 13.2, gate/up 28672 40.7 / 40.0; of 2048, N 4096 8.3 / 6.6, 32000 24.5 / 22.8, gate/up 16384 15.7 / 13.7; two of 2048, N 1024 8.3 / 6.8, 4096 8.4 / 8.1, 6144
  // 9.5 / 9.9, 12304 12.6 / 13.7; four of 512, N 4096 5.6 / 3.9, 32000 13.0 / 10.5; eight of 256 5.1 / 3.8, 9.6 / 7.6; five of 192 4.7 / 3.5, 8.4 / 7.1; sixteen of 256,
  // N 1024 5.0 / 4.6, 4096 5.4 / 5.2.  fp32: eight of 256, N 4096 5.9 / 4.1, 32000 15.3 / 13.4; one of 2048 10.6 / 8.4, 46 / 43; one of 4096, N 8192 27.7 / 27.1, but
  // 9000 30.1 / 34.8 (its product is bound by the matrix pipes, and the four waves of a unit of which it has one workgroup are too few for them).
  const bool dual = epi_dual(epi);
  if (sets > 8 && ((T > 1 && N > 4096) || (eb == 4 && !dual && N > 8192))) return 0;
  const LinExt ext = lin_dense(N, K);
  const bool ring = stream_ok(w, w, N, K, epi, ext, eb) && stream_pays(T, N, K, epi, 1, eb);
  // A pair's rows are twice the sums and four barriers: formed for every 16 rows of weights (the one-tile kernel, and a ring whose K is too short to run on) they
  // are more than the seam's launch from 8192 rows of weights on, of single matrices and 384 elements from 12288.  16 bits: one row of 64, 9168 5.6 / 6.5, 21536
  // 7.0 / 9.9; of 192, 33520 10.1 / 14.6; of 384, 10400 7.5 / 7.9 in four slabs, 1.05 ahead in the mean there, two rows, 23792 10.8 / 12.8; of 768, 39120 19.6 / 24.2;
  // gate/up, two of 64, 14272 6.8 / 8.3; fp32, one of 128, 10768 7.5 / 9.2, 38256 14.0 / 23.2.
  if (f->kind == UMB_FRONT_PAIR && N > (!dual && eb == 2 && K >= 384 ? 12288 : 8192) && (!ring || (long)K * eb < 3 * 512)) return 0;
  if (ring) return 1;
  // The one-tile kernel forms the rows for every 16 rows of weights, however many workgroups a unit works through.  16-bit weights of few steps are read in less than
  // that takes: one row of 1000, 16400 10.5 / 9.9, 24000 12.8 / 13.2, 128256 45 / 54; of 1536, 12304 12.5 / 11.8, 20000 14.9 / 15.2; of 640, 128256 39.5 / 33.5; two
  // of 768, 65536 24.3 / 23.2, 128256 41.1 / 42.7; gate/up of 512, 16384 11.3 / 10.6, 32768 15.8 / 15.8 (four rows 16.3 / 16.9).  fp32: 139 / 96 for two of 1000, N 128256.
  if (eb == 2 && N > 16384 && K >= (dual ? 512 : 641) && (dual || K > 768 || N > 65536)) return 0;
  return K <= (dual ? 1024 : 2048) ? 2 : 0;
}

extern "C" int umb_seq_front_ok(const UmbSeqFront* f, const void* w, int T, int N, int epi, int dtype) {
  return (dtype == UMB_SEQ_BF16 || dtype == UMB_SEQ_F16 || dtype == UMB_SEQ_F32) && front_form(f, w, T, N, epi, dtype) > 0;
}

template <typename P, bool DUAL, int KIND, int SETS>
static int launch_front_as(int form, void* out, float* x_out, const UmbSeqFront& f, const void* w, const void* bias, int T, int N, int epi, float limit, float alpha,
                        hipStream_t st) {
  typedef typename El<P>::type E;
  const int K = f.W, blocks = (N + 15) / 16;
  const size_t rows = (size_t)T * (K * sizeof(E) + 64);
  if (form == 1) {
    const int nc = (int)(K * sizeof(E) / 512);
    // slots and workgroups as in launch_stream; more blocks than those run on inside one workgroup a unit, whose rows are formed once, or two of fp32 (one and
    // two, us: four rows of 512, N 12304 9.8 / 8.4, 32000 18.2 / 14.4, the seam and the product 16.5; one of 2048 22.1 / 19.2, 43.6 / 42.3, 46.0)
#define FRONT_STREAM(SLOTS, RUN, GRID)                                                                                                                   do {                                                                                                                                                     const size_t lds = FrontRing<DUAL, SLOTS>::R * FrontRing<DUAL, SLOTS>::SLOT + rows;                                                                   if (ensure_dynamic_lds<front_stream_kernel<P, DUAL, KIND, SETS, SLOTS, RUN>>(lds) != UMB_OK) return UMB_EHIP;                                         hipLaunchKernelGGL((front_stream_kernel<P, DUAL, KIND, SETS, SLOTS, RUN>), dim3(GRID), dim3(512), lds, st, out, (const E*)w, (const E*)bias, T, N, K, epi,                        limit, alpha, GRID, nc >= 8 ? 7 : 0, x_out, f);                                                                                   } while (0)
    if constexpr (DUAL) {
      if (blocks > 400 && nc >= 3) FRONT_STREAM(3, true, 256);
      else FRONT_STREAM(3, false, blocks);
    } else {
      if (blocks > 512 && nc >= 5 && sizeof(E) == 2) FRONT_STREAM(5, true, 256);
      else if (blocks > 512 && nc >= 3) FRONT_STREAM(3, true, sizeof(E) == 2 ? 256 : 512);
      else if (blocks > 256) FRONT_STREAM(3, false, blocks);
      else FRONT_STREAM(4, false, blocks);
    }
#undef FRONT_STREAM
    UMB_LAUNCH_CHECK();
    return UMB_OK;
  }
#define FRONT_LINEAR(UN) \
  hipLaunchKernelGGL((front_linear_kernel<P, DUAL, KIND, SETS, UN>), dim3(blocks), dim3(256), rows, st, out, (const E*)w, (const E*)bias, T, N, K, epi, limit, alpha, x_out, f)
  if (K <= 256) FRONT_LINEAR(2);
  else if (K <= 512) FRONT_LINEAR(4);
  else if (DUAL || K <= 1024) FRONT_LINEAR(8);
  else if constexpr (!DUAL) FRONT_LINEAR(16);
#undef FRONT_LINEAR
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

template <typename P, bool DUAL, int KIND>
static int launch_front(int form, void* out, float* x_out, const UmbSeqFront& f, const void* w, const void* bias, int T, int N, int epi, float limit, float alpha,
                        hipStream_t st) {
  const int groups = KIND == UMB_FRONT_SEAM || KIND == UMB_FRONT_EMBED ? f.groups : 1, gs = f.W / groups;
  if (T * groups * ((gs + 255) / 256) <= 8) return launch_front_as<P, DUAL, KIND, 2>(form, out, x_out, f, w, bias, T, N, epi, limit, alpha, st);
  if constexpr (KIND == UMB_FRONT_PAIR && sizeof(typename El<P>::type) == 4) return UMB_EINVAL;
  else return launch_front_as<P, DUAL, KIND, 4>(form, out, x_out, f, w, bias, T, N, epi, limit, alpha, st);
}

extern "C" int umb_seq_front_linear(void* out, float* x_out, const UmbSeqFront* f, const void* w, const void* bias, int T, int N, int epi, float limit, float alpha,
                                    int dtype, hipStream_t st) {
  if (!out || !x_out || (uintptr_t)x_out % 16 || !f || x_out == f->x || !umb_seq_front_ok(f, w, T, N, epi, dtype) ||
      ((epi == EPI_CLAMP_GLU || epi == EPI_CAP) && !(limit > 0.f)))
    return UMB_EINVAL;
  const int form = front_form(f, w, T, N, epi, dtype), rows = epi_dual(epi) ? N / 2 : N;
#define FRONT(KIND)                                                                                                          \
  case KIND:                                                                                                                 \
    DISPATCH_SEQ_DTYPE(dtype, {                                                                                              \
      return epi_dual(epi) ? launch_front<P, true, KIND>(form, out, x_out, *f, w, bias, T, rows, epi, limit, alpha, st)      \
                           : launch_front<P, false, KIND>(form, out, x_out, *f, w, bias, T, rows, epi, limit, alpha, st);    \
    })
  switch (f->kind) {
    FRONT(UMB_FRONT_SEAM)
    FRONT(UMB_FRONT_STREAM)
    FRONT(UMB_FRONT_PAIR)
    FRONT(UMB_FRONT_EMBED)
    default: return UMB_EINVAL;
  }
#undef FRONT
}
