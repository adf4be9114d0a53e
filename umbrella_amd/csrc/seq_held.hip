// Streaming products of 33 to 64 tokens whose tokens stay in registers (the others: seq_linear.hip).
//
// A workgroup of the streaming kernel fetches its chunk of the tokens again beside every block of weight rows: 24 to 32 KiB of them beside 16, from L2, but
// in the same ring, whose two chunks ahead are all that LDS holds of both -- some 80 KB under way in a unit, a third of them weights.  Here a workgroup that has
// several blocks of rows keeps what its waves read of the tokens in the first one: K / 4 of each, 192 to 384 registers, which one workgroup a unit leaves
// to a wave.  From the second block on only weights are fetched, four chunks ahead.
// us, bf16, cold weights, the streaming kernel / this: 48 tokens 32000 x 2048 31.3 / 26.8 (4.9 TB/s of weights), x 4096 53.7 / 49.4, gate/up 14336 x 4096 52.1 / 43.5,
// 8192 x 2048 17.0 / 16.7, 5120 x 2048 16.0 / 15.0; 10240 x 2048 16.6 / 15.2; 64 tokens 32000 x 2048 36.8 / 29.4, gate/up 8192 x 2048
// 19.6 / 18.5, 14336 x 4096 59.1 / 50.3 (ten of the sixteen chunks of 4096 stay: more are more than a wave's registers), 32000 x 4096 62.6 / 54.5; other K: held_pays.
// The arithmetic is the streaming kernel's, sum for sum: chunks from the same place on (a workgroup's blocks are 4096 rows and more apart, so that they all
// begin with the same one), the same wave for the same 32 k, the waves' tiles added in the same order.
#include "seq_linear.h"

template <int C, int N, typename F> __device__ __forceinline__ void unrolled(F f) {
  if constexpr (C < N) {
    f(std::integral_constant<int, C>{});
    unrolled<C + 1, N>(f);
  }
}

// slots of the weights' ring and, for the first block, of the tokens'
template <int NT, int TT, bool DUAL> struct HeldShape {
  typedef StreamShape<NT, TT, 8 * TT, DUAL, 2> S;
  static constexpr int AP = S::AP, BP = 8 * TT, AT = S::AT, PA = AP / 4, PB = BP / 4, RB = TT == 3 ? 3 : 2, RA = 5;
  static constexpr unsigned PIECE = S::PIECE, SLOT_A = AP * PIECE, SLOT_B = BP * PIECE, TOKENS = RA * SLOT_A;
  static constexpr size_t LDS = TOKENS + RB * SLOT_B;
  static_assert(LDS <= 160 * 1024 && S::RED <= RB * SLOT_B && RA >= RB, "the unit's LDS; the waves' tiles in the tokens' ring");
};
// K: 5 to MC chunks.  HC: those whose tokens stay, from the first on; the others' are fetched with every block's
template <typename P, int NT, int TT, bool DUAL, int MC, int HC>
__global__ __launch_bounds__(256, 1) void held_stream_kernel(void* __restrict__ out_, const u16* __restrict__ x, const u16* __restrict__ w,
                                                             const u16* __restrict__ bias, int T, int N, int K, int epi, float limit, float alpha) {
  typedef HeldShape<NT, TT, DUAL> H;
  constexpr int STEP = 256, AT = H::AT, PA = H::PA, PB = H::PB, RA = H::RA, RB = H::RB;
  constexpr unsigned PIECE = H::PIECE, SLOT_A = H::SLOT_A, SLOT_B = H::SLOT_B;
  static_assert(HELD_MIN >= RA && HC >= RB && STEP * 16 % 1024 == 0, "a ring's chunks are of two blocks at most; blocks that begin with the same chunk");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, g = lane >> 4;
  const unsigned lds0 = (unsigned)(size_t)(lds_char*)smem, lds1 = lds0 + H::TOKENS;
  const int odd = lane >> 5, c16 = ((lane & 31) ^ (odd * 8)) * 16;
  unsigned va[PA], vb[PB];                                   // pieces of two rows, as in the streaming kernel
  auto rows_of_block = [&](int n0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int r = 2 * (wave + 4 * i) + odd, n = DUAL && r >= 16 * NT ? N + min(n0 + r - 16 * NT, N - 1) : min(n0 + r, N - 1);
      va[i] = (unsigned)(n - n0) * (unsigned)(K * 2) + c16;
    }
  };
#pragma unroll
  for (int i = 0; i < PB; ++i) vb[i] = (unsigned)min(2 * (wave + 4 * i) + odd, T - 1) * (unsigned)(K * 2) + c16;
  const int nc = K / 256, nb = (N + 16 * NT - 1) / (16 * NT), start = first_chunk(blockIdx.x * (16 * NT), nc, nc >= 8 ? 7 : 0);
  const char* wb = reinterpret_cast<const char*>(w);
  const char* xb = reinterpret_cast<const char*>(x);
  int fb = blockIdx.x, col = start, left = nc;               // the block whose weights are fetched, its next chunk, those still to come
  const char* fw = wb + (long)fb * (16 * NT) * K * 2;
  rows_of_block(fb * (16 * NT));
  auto weights = [&](int slot) __attribute__((always_inline)) {
    const long at = (long)col * 512;
#pragma unroll
    for (int i = 0; i < PA; ++i) tile_dma_once(va[i], fw + at, lds0 + (unsigned)slot * SLOT_A + (unsigned)(wave + 4 * i) * PIECE);
    col = col + 1 == nc ? 0 : col + 1;
    if (--left == 0 && fb + STEP < nb) {                     // behind the last block its chunks are fetched again, never read
      fb += STEP;
      left = nc;
      fw = wb + (long)fb * (16 * NT) * K * 2;
      rows_of_block(fb * (16 * NT));
    }
  };
  auto tokens = [&](int c) __attribute__((always_inline)) {
    const long at = (long)(start + c < nc ? start + c : start + c - nc) * 512;
#pragma unroll
    for (int i = 0; i < PB; ++i) tile_dma(vb[i], xb + at, lds1 + (unsigned)(c % RB) * SLOT_B + (unsigned)(wave + 4 * i) * PIECE);
  };
  const unsigned row = H::S::row_at(0, 8, j), swz = (unsigned)(j & 1) * 8u;
  auto frag = [&](unsigned base, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const lds_u32x4*>((size_t)(base + row + (((unsigned)(s * 4 + g)) ^ swz) * 16u));
  };
  u32x4 held[HC][2][TT];                                     // this wave's tokens: two steps of 32 k of a chunk
  f32x4 acc[AT][TT];
  int slot = 0;
  auto chunk = [&](auto c_, auto first_) __attribute__((always_inline)) {
    constexpr int c = decltype(c_)::value;
    constexpr bool first = decltype(first_)::value, fetched = first || c >= HC;
    // what was asked for behind this chunk's last piece: its tokens', with RB - 1 chunks of weights and RB - 2 of tokens behind (none behind the last
    // chunk's), or its weights'
    static_assert(RB <= 3);
    if constexpr (!fetched) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((RA - 2) * PA) : "memory");
    else if (RB == 3 && c + 1 == nc) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((RB - 1) * PA) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((RB - 1) * PA + (RB - 2) * PB) : "memory");
    __builtin_amdgcn_s_barrier();
    if constexpr (first || c + RB - 1 >= HC)
      if (c + RB - 1 < nc) tokens(c + RB - 1);
    weights(slot == 0 ? RA - 1 : slot - 1);
    const unsigned base = lds0 + (unsigned)slot * SLOT_A;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int s = wave + 4 * u;
      u32x4 a[AT];
#pragma unroll
      for (int i = 0; i < AT; ++i) a[i] = frag(base + (unsigned)(8 * i) * PIECE, s);
      u32x4 t[TT];
      if constexpr (fetched) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) t[tt] = frag(lds1 + (unsigned)(c % RB) * SLOT_B + (unsigned)(8 * tt) * PIECE, s);
      }
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        if constexpr (first && c < HC) held[c][u][tt] = t[tt];
        if constexpr (!fetched) t[tt] = held[c][u][tt];
      }
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int i = 0; i < AT; ++i) acc[i][tt] = P::mfma(a[i], t[tt], acc[i][tt]);
    }
    slot = slot + 1 == RA ? 0 : slot + 1;
  };
  auto block = [&](int b, auto first_) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AT; ++i)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) acc[i][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    unrolled<0, MC>([&](auto c_) __attribute__((always_inline)) {
      if (decltype(c_)::value < HELD_MIN || decltype(c_)::value < nc) chunk(c_, first_);
    });
    // the waves' tiles are added in the tokens' ring: nobody reads it behind a block's last chunk, and its pieces are asked for again behind the next's first
    if (b + STEP >= nb) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // behind the last block no piece may be on its way any more
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < AT; ++i)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) *reinterpret_cast<lds_f32x4*>((size_t)(lds1 + (((wave * AT + i) * TT + tt) * 256 + lane * 4) * 4u)) = acc[i][tt];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const int l = threadIdx.x >> 2, r = threadIdx.x & 3;
    auto total = [&](int i, int tt) __attribute__((always_inline)) {
      const auto at = [&](int ww) { return *reinterpret_cast<const lds_f32*>((size_t)(lds1 + (((ww * AT + i) * TT + tt) * 256 + threadIdx.x) * 4u)); };
      float s = at(0);
#pragma unroll
      for (int ww = 1; ww < 4; ++ww) s += at(ww);
      return s;
    };
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = b * 16 * NT + nt * 16 + 4 * (l >> 4) + r;
      if (n >= N) continue;
      const float bv = bias ? ldf<P>(bias + n) : 0.f, bv2 = (DUAL && bias) ? ldf<P>(bias + N + n) : 0.f;
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const int t = tt * 16 + (l & 15);
        if (t >= T) continue;
        const float s = total(nt, tt) + bv;
        const long o = (long)t * N + n;
        if constexpr (DUAL) stf<P>(reinterpret_cast<u16*>(out_) + o, glu_pair(epi, s, total(NT + nt, tt) + bv2, limit, alpha));
        else if (epi == EPI_DT) stf<P>(reinterpret_cast<u16*>(out_) + o, s);
        else if (epi == EPI_RELU2) {
          const float rl = fmaxf(s, 0.f);
          stf<P>(reinterpret_cast<u16*>(out_) + o, rl * rl);
        }
        else if (epi == EPI_CAP) reinterpret_cast<float*>(out_)[o] = limit * tanhf(s / limit);
        else reinterpret_cast<float*>(out_)[o] = s;
      }
    }
  };
#pragma unroll
  for (int c = 0; c < RA - 1; ++c) {
    weights(c);
    if (c < RB - 1) tokens(c);
  }
  block(blockIdx.x, std::true_type{});
  for (int b = blockIdx.x + STEP; b < nb; b += STEP) block(b, std::false_type{});
}

template <typename P, int NT, int TT, bool DUAL, int MC, int HC = MC>
static int held_launch(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, float limit, float alpha, hipStream_t st) {
  constexpr size_t lds = HeldShape<NT, TT, DUAL>::LDS;
  if (ensure_dynamic_lds<held_stream_kernel<P, NT, TT, DUAL, MC, HC>>(lds) != UMB_OK) return UMB_EHIP;
  hipLaunchKernelGGL((held_stream_kernel<P, NT, TT, DUAL, MC, HC>), dim3(256), dim3(256), lds, st, out, (const u16*)x, (const u16*)w, (const u16*)bias, T, N, K,
                     epi, limit, alpha);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

int held_stream(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, float limit, float alpha, int dtype, hipStream_t st) {
  if (!held_pays(T, N, K, epi)) return UMB_EINVAL;
  auto run = [&](auto tag) -> int {
    typedef decltype(tag) P;
#define HELD(TT, ...) (epi_dual(epi) ? held_launch<P, 1, TT, true, __VA_ARGS__>(out, x, w, bias, T, N, K, epi, limit, alpha, st) \
                                     : held_launch<P, 2, TT, false, __VA_ARGS__>(out, x, w, bias, T, N, K, epi, limit, alpha, st))
    // (eight chunks by themselves: half of the code, all of whose loads are fetched)
    if (T <= 48) return K <= 8 * 256 ? HELD(3, 8) : HELD(3, 16);
    return K <= 8 * 256 ? HELD(4, 8) : HELD(4, 16, 10);
#undef HELD
  };
  return dtype == UMB_SEQ_BF16 ? run(BF16{}) : dtype == UMB_SEQ_F16 ? run(F16{}) : UMB_EINVAL;
}
