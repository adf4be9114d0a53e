// General linear layer for the sequence-mixer models: out[T][N] = x[T][K] . W[N][K]^T + bias for ANY T, N, K, weights as
// stored (row-major [out][in], no repacking), 16-bit or fp32 storage, fp32 accumulation on the matrix pipe.
//
// Both operands are K-contiguous, so a lane's 8 consecutive K-elements of "its" row ARE its share of an MFMA operand:
//   v_mfma_f32_16x16x32_{bf16,f16}: A 16 rows x 32 k, lane (j = lane % 16, g = lane / 16) supplies row j, k 8g .. 8g+7
//   v_mfma_f32_16x16x4_f32 (true fp32, x8): the same 8 elements feed instruction i with element i of every lane, i.e. step i
//   multiplies k = 8g + i of A with k = 8g + i of B -- the pairing is what matters, the order inside the 32-k step is free.
// Weights are the A operand (rows = output features), tokens the B operand: lane l ends up with outputs
// (n = 4 (l / 16) + r, token = l % 16), r = 0..3.  Weights go HBM -> VGPR (every weight element is used by exactly one wave of
// a <= 64-token launch), as in the skinny GEMM of gemm.hip.
//
// Few tokens: a workgroup owns 16 (or 32) output rows and up to 64 tokens; its four waves split K (wave w takes the 32-k steps w, w+4, ...)
// and their partial tiles are summed through LDS in wave order: the summation order of an output is a function of K and of its row of W,
// never of the token's place in the batch, and of T only where the many-token kernels take over (launch_vec).  K % 8 != 0 (or a tail)
// falls back to guarded element loads.
#include "seq_linear.h"
#include <algorithm>

// NT output tiles x TT token tiles of 16 per workgroup (each wave holds all NT x TT accumulator tiles of its K share: one weight
// fragment meets TT token fragments and one token fragment NT weight fragments, so a launch of many tokens moves
// 1 / NT + 1 / TT fragment loads per MFMA instead of 1 + 1 / TT); DUAL: a second weight matrix W2 = W + N * K (the "up" half)
// with its own accumulators (NT <= 2: the partial tiles of both halves share the 64 KiB of LDS).
template <typename P, int NT, int TT, bool VEC, bool DUAL>
__global__ __launch_bounds__(256) void seq_linear_kernel(void* __restrict__ out_, const typename El<P>::type* __restrict__ x,
                                                         const typename El<P>::type* __restrict__ w,
                                                         const typename El<P>::type* __restrict__ bias, int T, int N, int K,
                                                         int epi, LinExt ext) {
  typedef typename El<P>::type E;
  static_assert(!DUAL || NT <= 2, "gate and up partials of NT x TT tiles must fit the LDS");
  __shared__ float red[DUAL ? 2 : 1][4][NT * TT][256];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int j = lane & 15, g = lane >> 4;
  int t0 = blockIdx.y * (TT * 16);
  const int ldx = ext.ldx, ldo = ext.ldo;
  long obase = (long)blockIdx.z * ext.so;
  const float* gate = ext.gate ? ext.gate + (long)blockIdx.z * ext.sg : nullptr;
  x += (long)blockIdx.z * ext.sx;
  w += (long)blockIdx.z * ext.sw;
  if (ext.tiles) {                         // grouped: this workgroup's rows and weights come from the tile list
    const int* td = ext.tiles + 3 * blockIdx.y;
    const int rows = td[2];
    if (rows <= 0) return;
    w += (long)td[0] * ext.gs;
    x += (long)td[1] * ldx;
    obase += (long)td[1] * ldo;
    T = rows;
    t0 = 0;
  }
  const E* wrow[NT];                       // rows past an operand's end read its last one: what they give is not stored
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) wrow[nt] = w + (long)min((int)(blockIdx.x * NT + nt) * 16 + j, N - 1) * K;
  const long half = DUAL ? (long)N * K : 0;
  const E* xrow[TT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) xrow[tt] = x + (long)min(t0 + tt * 16 + j, T - 1) * ldx;
  // thread (l = tid / 4, r = tid % 4) finishes output (n = 4 (l / 16) + r, token = l % 16) of every tile; its biases are asked for beside the
  // operands: behind the sums they were a round trip of their own
  const int l = threadIdx.x >> 2, r = threadIdx.x & 3;
  float bv[NT], bv2[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = min((int)(blockIdx.x * NT + nt) * 16 + 4 * (l >> 4) + r, N - 1);
    bv[nt] = bias ? ldf<P>(bias + n) : 0.f;
    bv2[nt] = (DUAL && bias) ? ldf<P>(bias + N + n) : 0.f;
  }
  f32x4 acc[NT][TT], acc2[NT][TT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) { acc[nt][tt] = f32x4{0.f, 0.f, 0.f, 0.f}; acc2[nt][tt] = f32x4{0.f, 0.f, 0.f, 0.f}; }
  }

  // this wave's 32-k steps k0, k0 + 128, ...: `un` of them in flight at once.  (A step past K is zeros; the loads and, in fp32, eight products of it
  // cost as much as any other's, see UN.)
  auto steps = [&](auto un, int k0) __attribute__((always_inline)) {
    constexpr int U = decltype(un)::value;
    Frag8<P> a[U][NT], a2[U][NT], b[U][TT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 128 + g * 8;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        a[u][nt] = load8<P, VEC>(wrow[nt], k, K);
        if constexpr (DUAL) a2[u][nt] = load8<P, VEC>(wrow[nt] + half, k, K);
      }
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) b[u][tt] = load8<P, VEC>(xrow[tt], k, K);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc[nt][tt] = mma8<P>(a[u][nt], b[u][tt], acc[nt][tt]);
          if constexpr (DUAL) acc2[nt][tt] = mma8<P>(a2[u][nt], b[u][tt], acc2[nt][tt]);
        }
      }
    }
  };
  // A single tile's launch is latency-bound: all its steps in flight, up to 16 (8 of both halves), K = 2048 in one round trip.  The last ones by the
  // least power of two that holds them: as 16 whatever K is, K = 192 in fp32 was fourteen steps of zeros, 112 of 128 products.
  constexpr int UN = (NT * TT == 1) ? (DUAL ? 8 : 16) : 2;
  int k0 = wave * 32;
  for (; K - k0 > 128 * (UN / 2); k0 += 128 * UN) steps(std::integral_constant<int, UN>{}, k0);
  if constexpr (UN > 8) if (K - k0 > 128 * 4) { steps(std::integral_constant<int, 8>{}, k0); k0 = K; }
  if constexpr (UN > 4) if (K - k0 > 128 * 2) { steps(std::integral_constant<int, 4>{}, k0); k0 = K; }
  if constexpr (UN > 2) if (K - k0 > 128) { steps(std::integral_constant<int, 2>{}, k0); k0 = K; }
  if (K > k0) steps(std::integral_constant<int, 1>{}, k0);
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      *reinterpret_cast<f32x4*>(&red[0][wave][nt * TT + tt][lane * 4]) = acc[nt][tt];
      if constexpr (DUAL) *reinterpret_cast<f32x4*>(&red[1][wave][nt * TT + tt][lane * 4]) = acc2[nt][tt];
    }
  }
  __syncthreads();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = (blockIdx.x * NT + nt) * 16 + 4 * (l >> 4) + r;
    if (n >= N) continue;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      const int t = t0 + tt * 16 + (l & 15);
      if (t >= T) continue;
      float s = red[0][0][nt * TT + tt][threadIdx.x];
#pragma unroll
      for (int ww = 1; ww < 4; ++ww) s += red[0][ww][nt * TT + tt][threadIdx.x];
      s += bv[nt];
      if constexpr (DUAL) {
        float u = red[1][0][nt * TT + tt][threadIdx.x];
#pragma unroll
        for (int ww = 1; ww < 4; ++ww) u += red[1][ww][nt * TT + tt][threadIdx.x];
        u += bv2[nt];
        stf<P>(reinterpret_cast<E*>(out_) + obase + (long)t * ldo + n, glu_pair(epi, s, u, ext.limit, ext.alpha));
      } else if (epi == EPI_DT) {
        stf<P>(reinterpret_cast<E*>(out_) + obase + (long)t * ldo + n, s);
      } else if (epi == EPI_RELU2) {
        const float rl = fmaxf(s, 0.f);
        stf<P>(reinterpret_cast<E*>(out_) + obase + (long)t * ldo + n, rl * rl);
      } else if (epi == EPI_GATE) {
        stf<P>(reinterpret_cast<E*>(out_) + obase + (long)t * ldo + n, s / (1.f + expf(-gate[(long)t * ext.ldg + n])));
      } else if (epi == EPI_GATE_ROW) {
        stf<P>(reinterpret_cast<E*>(out_) + obase + (long)t * ldo + n, s / (1.f + expf(-gate[(long)t * ext.ldg])));
      } else if (epi == EPI_CAP) {
        reinterpret_cast<float*>(out_)[obase + (long)t * ldo + n] = ext.limit * tanhf(s / ext.limit);
      } else {
        reinterpret_cast<float*>(out_)[obase + (long)t * ldo + n] = s;
      }
    }
  }
}

// ---- many tokens (T > 64), 16-bit storage: a 128 x 128 output tile per workgroup, operands staged through LDS.
// The skinny kernel above streams every weight once per 64 tokens and every token fragment once per 16 (or 64) output rows
// straight from L2: right when weights dominate, wasteful when both operands are re-used 128 times.  Here a stage of 64 k
// (A: 128 output rows, B: 128 tokens, 16 KiB each) is fetched with 16-byte loads into registers while the previous stage is
// consumed, written to the other half of a double-buffered 64 KiB LDS tile, and each of the four waves (2 x 2) reads the
// fragments of its 64 x 64 sub-tile from there: 8 fragment reads per 16 MFMAs, every read a contiguous KiB (the tile is
// stored as two [128 rows][32 k] halves so that a fragment's 16 rows x 64 B are adjacent: no bank conflict).
// K is summed in order inside one accumulator (no K split): results differ from the skinny kernel by rounding only.
// DUAL (gate/up): the 128 staged weight rows are 64 gate rows and the 64 up rows of the same outputs.
template <typename P, bool DUAL>
__global__ __launch_bounds__(256) void seq_linear_wide_kernel(void* __restrict__ out_, const u16* __restrict__ x,
                                                              const u16* __restrict__ w, const u16* __restrict__ bias, int T,
                                                              int N, int K, int epi, LinExt ext) {
  __shared__ __attribute__((aligned(16))) u16 tile[2][2][2][128 * 32];      // [buffer][A | B][k half][row][32 k]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  int t0 = blockIdx.y * 128;
  long obase = 0;
  if (ext.tiles) {                         // grouped: a tile of up to 128 rows of one group
    const int* td = ext.tiles + 3 * blockIdx.y;
    if (td[2] <= 0) return;
    w += (long)td[0] * ext.gs;
    x += (long)td[1] * K;
    obase = (long)td[1] * N;
    T = td[2];
    t0 = 0;
  }
  const int n0 = blockIdx.x * (DUAL ? 64 : 128);
  // staging: thread owns chunks c = tid + 256 i (i < 4) of each operand's 128 x 8 chunk grid: row c / 8, 16-byte chunk c % 8
  const u16* asrc[4];
  const u16* bsrc[4];
  bool aok[4], bok[4];
  int soff[4], kc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + 256 * i, row = c >> 3, ch = c & 7;
    int n = DUAL ? (row < 64 ? n0 + row : N + n0 + (row - 64)) : n0 + row;
    aok[i] = DUAL ? (n0 + (row & 63) < N) : (n < N);
    asrc[i] = w + (long)(aok[i] ? n : 0) * K + ch * 8;
    bok[i] = t0 + row < T;
    bsrc[i] = x + (long)(bok[i] ? t0 + row : 0) * K + ch * 8;
    kc[i] = ch * 8;
    soff[i] = (ch >> 2) * (128 * 32) + row * 32 + (ch & 3) * 8;
  }
  u32x4 ra[4], rb[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = k0 + kc[i] < K;
      ra[i] = (aok[i] && in) ? *reinterpret_cast<const u32x4*>(asrc[i] + k0) : u32x4{0u, 0u, 0u, 0u};
      rb[i] = (bok[i] && in) ? *reinterpret_cast<const u32x4*>(bsrc[i] + k0) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<u32x4*>(&tile[buf][0][0][0] + soff[i]) = ra[i];
      *reinterpret_cast<u32x4*>(&tile[buf][1][0][0] + soff[i]) = rb[i];
    }
  };
  int arow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) arow[i] = DUAL ? ((i >> 1) * 64 + wm * 32 + (i & 1) * 16) : (wm * 64 + i * 16);
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) acc[i][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  stash(0);
  __syncthreads();
  const int nst = (K + 63) / 64;
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1;
    if (st + 1 < nst) fetch((st + 1) * 64);
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      u32x4 fa[4], fb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        fa[i] = *reinterpret_cast<const u32x4*>(&tile[buf][0][kh][(arow[i] + j) * 32 + g * 8]);
        fb[i] = *reinterpret_cast<const u32x4*>(&tile[buf][1][kh][(wn * 64 + i * 16 + j) * 32 + g * 8]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) acc[i][tt] = P::mfma(fa[i], fb[tt], acc[i][tt]);
    }
    if (st + 1 < nst) stash(buf ^ 1);
    __syncthreads();
  }
  // lane holds outputs (row = 4 g + r of its A tile, token = j of its B tile)
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    const int t = t0 + wn * 64 + tt * 16 + j;
    if (t >= T) continue;
#pragma unroll
    for (int i = 0; i < (DUAL ? 2 : 4); ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + (DUAL ? wm * 32 + i * 16 : arow[i]) + 4 * g + r;
        if (n >= N) continue;
        float sv = acc[i][tt][r] + (bias ? P::to_f(bias[n]) : 0.f);
        if constexpr (DUAL) {
          const float uv = acc[i + 2][tt][r] + (bias ? P::to_f(bias[N + n]) : 0.f);
          reinterpret_cast<u16*>(out_)[obase + (long)t * N + n] = P::from_f(glu_pair(epi, sv, uv, ext.limit, ext.alpha));
        } else if (epi == EPI_DT) {
          reinterpret_cast<u16*>(out_)[obase + (long)t * N + n] = P::from_f(sv);
        } else if (epi == EPI_RELU2) {
          const float rl = fmaxf(sv, 0.f);
          reinterpret_cast<u16*>(out_)[obase + (long)t * N + n] = P::from_f(rl * rl);
        } else if (epi == EPI_CAP) {
          reinterpret_cast<float*>(out_)[obase + (long)t * N + n] = ext.limit * tanhf(sv / ext.limit);
        } else {
          reinterpret_cast<float*>(out_)[obase + (long)t * N + n] = sv;
        }
      }
    }
  }
}

// ---- many tokens, both operands dense with whole 64-k stages: the staged product of gemm_tile.h.  DUAL: a wave's RA row tiles are
// RA / 2 tiles of gate rows and the up rows of the same outputs.  The k order of an output without K-split is the wide kernel's:
// the same bits.
// A workgroup of the launch: tile number id of nbt token tiles a column, slab sp of K, the columns from row `first` on.
template <typename P, int WM, int WN, int RA, int RB, int KS, bool DUAL>
__device__ __forceinline__ void tile_block(unsigned char* smem, void* __restrict__ out_, const u16* __restrict__ x, const u16* __restrict__ w,
                                           const u16* __restrict__ bias, int T, int N, int K, int epi, int nbt, int slabs, float limit, float alpha,
                                           int tile, int sp, int first) {
  typedef TileShape<WM, WN, RA, RB, KS> S;
  constexpr int OUTN = DUAL ? S::BN / 2 : S::BN;
  const int lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_all % S::NW, ks = wave_all / S::NW, j = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
  const int column = __builtin_amdgcn_readfirstlane(tile / nbt), n0 = first + column * OUTN, t0 = (tile - column * nbt) * S::BT;
  // slab sp of K (one more stage in the first ones): its sums go to out + sp T N, the bias into slab 0's
  const int each = __builtin_amdgcn_readfirstlane(K / 64 / slabs), longer = K / 64 - each * slabs, st0 = sp * each + min(sp, longer), stages = each + (sp < longer);
  // rows past the operand's end re-read its last row: their outputs are not stored
  unsigned voff[S::NPW];
#pragma unroll
  for (int i = 0; i < S::NPW; ++i) {
    const int p = wave + S::NW * i;
    if (S::NW * i < S::NPA)
      voff[i] = tile_voff(p, lane, K, [&](int row) {
        if (!DUAL) return min(n0 + row, N - 1) - n0;
        const int h = row / (16 * RA), in = row % (16 * RA), up = in / (8 * RA), rr = in % (8 * RA);
        return min(n0 + h * (8 * RA) + rr, N - 1) - n0 + up * N;
      });
    else voff[i] = tile_voff(p - S::NPA, lane, K, [&](int row) { return min(t0 + row, T - 1) - t0; });
  }
  f32x4 acc[RA][RB];
  if (!tile_products<P, WM, WN, RA, RB, KS, false>(acc, smem, w + (long)n0 * K + st0 * 64, x + (long)t0 * K + st0 * 64, 128, voff, stages, wave, ks))
    return;
  if (sp) {
    out_ = reinterpret_cast<float*>(out_) + (long)sp * T * N;
    bias = nullptr;
  }
  constexpr int NI = DUAL ? RA / 2 : RA;
  const int nw = n0 + (DUAL ? wm * (8 * RA) : wm * (16 * RA));         // this wave's first output
  const bool half = DUAL || epi == EPI_DT || epi == EPI_RELU2;                 // 16-bit outputs
  const unsigned strip = (unsigned)(size_t)(lds_char*)smem + (unsigned)wave * (KS == 2 ? RA * RB * 1024u : TileRows<16, RA>::BYTES);
  static_assert(TileRows<16, RA>::BYTES <= RA * RB * 1024u && TileRows<16, RA>::BYTES * S::NW <= S::LDS, "a strip per wave");
  float bv[NI][4], bu[NI][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int nn = min(nw + i * 16 + 4 * g + r, N - 1);
      bv[i][r] = bias ? P::to_f(bias[nn]) : 0.f;
      bu[i][r] = DUAL && bias ? P::to_f(bias[N + nn]) : 0.f;
    }
  auto finish = [&](auto form) __attribute__((always_inline)) {      // (one copy of the loop for each epilogue: no tests inside)
  constexpr int EPI = decltype(form)::value;
#pragma unroll
  for (int t = 0; t < RB; ++t) {
    const int tile0 = t0 + (wn * RB + t) * 16, tok = tile0 + j;
    f32x4 v[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float s = acc[i][t][r] + bv[i][r];
        if constexpr (DUAL) {
          s = glu_of<EPI>(s, acc[i + RA / 2][t][r] + bu[i][r], limit, alpha);
        } else if constexpr (EPI == EPI_RELU2) {
          const float rl = fmaxf(s, 0.f);
          s = rl * rl;
        } else if constexpr (EPI == EPI_CAP) {
          s = limit * tanhf(s / limit);
        }
        v[i][r] = s;
      }
    }
    if (half && N % 8 == 0) {                                // rows of whole 16-byte groups: whole lines at a time
      u32x2 d[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) d[i] = u32x2{pack2<P>(v[i][0], v[i][1]), pack2<P>(v[i][2], v[i][3])};
      tile_rows_out<8, NI>(strip, d, [&](int row, int at, u32x4 b) {
        if (tile0 + row < T && nw + at / 2 < N) *reinterpret_cast<u32x4*>(reinterpret_cast<u16*>(out_) + (long)(tile0 + row) * N + nw + at / 2) = b;
      });
      continue;
    }
    if (!DUAL && !half && N % 4 == 0) {
      tile_rows_out<16, NI>(strip, v, [&](int row, int at, u32x4 b) {
        if (tile0 + row < T && nw + at / 4 < N) *reinterpret_cast<u32x4*>(reinterpret_cast<float*>(out_) + (long)(tile0 + row) * N + nw + at / 4) = b;
      });
      continue;
    }
    if (tok >= T) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = nw + i * 16 + 4 * g;
      const long o = (long)tok * N + n;
      if (n < N && half && N % 4 == 0) {
        *reinterpret_cast<u32x2*>(reinterpret_cast<u16*>(out_) + o) = u32x2{pack2<P>(v[i][0], v[i][1]), pack2<P>(v[i][2], v[i][3])};
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (n + r >= N) continue;
        if (half) reinterpret_cast<u16*>(out_)[o + r] = P::from_f(v[i][r]);
        else reinterpret_cast<float*>(out_)[o + r] = v[i][r];
      }
    }
  }
  };
  if constexpr (DUAL) {
    if (epi == EPI_CLAMP_GLU) finish(std::integral_constant<int, EPI_CLAMP_GLU>{});
    else if (epi == EPI_GELU_MUL) finish(std::integral_constant<int, EPI_GELU_MUL>{});
    else finish(std::integral_constant<int, EPI_SILU_MUL>{});
  } else {
    if (epi == EPI_RELU2) finish(std::integral_constant<int, EPI_RELU2>{});
    else if (epi == EPI_CAP) finish(std::integral_constant<int, EPI_CAP>{});
    else finish(std::integral_constant<int, EPI_F32>{});
  }
}

template <typename P, int WM, int WN, int RA, int RB, int KS, bool DUAL>
__global__ __launch_bounds__(64 * WM * WN * KS, WM * WN * KS == 4 ? 2 : 1)
void seq_linear_tile_kernel(void* __restrict__ out, const u16* __restrict__ x, const u16* __restrict__ w, const u16* __restrict__ bias,
                            int T, int N, int K, int epi, int nbt, int slabs, float limit, float alpha) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // (quotients go through the vector pipe: named uniform, or the addresses built on them are not)
  const int id = tile_of_block(blockIdx.x, gridDim.x), tiles = __builtin_amdgcn_readfirstlane(gridDim.x / slabs), sp = __builtin_amdgcn_readfirstlane(id / tiles);
  tile_block<P, WM, WN, RA, RB, KS, DUAL>(smem, out, x, w, bias, T, N, K, epi, nbt, slabs, limit, alpha, id - sp * tiles, sp, 0);
}

// Whole rounds of 256 x 256 tiles (the first `whole` workgroups), then the columns that are left in tiles of fewer tokens (tile_mix): a last round of
// 256 x 256 tiles takes as long as the others however few it has.
template <typename P, int RB, bool DUAL>
__global__ __launch_bounds__(512, 1)
void seq_linear_mixed_kernel(void* __restrict__ out, const u16* __restrict__ x, const u16* __restrict__ w, const u16* __restrict__ bias,
                             int T, int N, int K, int epi, int nbt, int nbt_tail, int whole, int first, float limit, float alpha) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int b = blockIdx.x;
  if (b < whole) tile_block<P, 4, 2, 4, 8, 1, DUAL>(smem, out, x, w, bias, T, N, K, epi, nbt, 1, limit, alpha, tile_of_block(b, whole), 0, 0);
  else tile_block<P, 4, 2, 4, RB, 1, DUAL>(smem, out, x, w, bias, T, N, K, epi, nbt_tail, 1, limit, alpha, tile_of_block(b - whole, gridDim.x - whole), 0, first);
}

template <typename P, int RB, bool DUAL>
static int launch_mixed(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, int columns, float limit, float alpha,
                        hipStream_t st) {
  typedef TileShape<4, 2, 4, 8, 1> S;
  typedef TileShape<4, 2, 4, RB, 1> Tail;
  constexpr int OUTN = DUAL ? S::BN / 2 : S::BN;
  constexpr size_t LDS = S::LDS > Tail::LDS ? S::LDS : Tail::LDS;
  if (ensure_dynamic_lds<seq_linear_mixed_kernel<P, RB, DUAL>>(LDS) != UMB_OK) return UMB_EHIP;
  const int first = columns * OUTN, nbt = (T + S::BT - 1) / S::BT, nbt_tail = (T + Tail::BT - 1) / Tail::BT, whole = columns * nbt;
  hipLaunchKernelGGL((seq_linear_mixed_kernel<P, RB, DUAL>), dim3((unsigned)whole + (N - first + OUTN - 1) / OUTN * nbt_tail), dim3(512), LDS, st,
                     out, (const u16*)x, (const u16*)w, (const u16*)bias, T, N, K, epi, nbt, nbt_tail, whole, first, limit, alpha);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

template <typename P, int WM, int WN, int RA, int RB, int KS, bool DUAL>
static int launch_tile_as(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, int slabs, float limit,
                          float alpha, hipStream_t st) {
  typedef TileShape<WM, WN, RA, RB, KS> S;
  constexpr int OUTN = DUAL ? S::BN / 2 : S::BN;
  if (ensure_dynamic_lds<seq_linear_tile_kernel<P, WM, WN, RA, RB, KS, DUAL>>(S::LDS) != UMB_OK) return UMB_EHIP;
  const int nbn = (N + OUTN - 1) / OUTN, nbt = (T + S::BT - 1) / S::BT;
  hipLaunchKernelGGL((seq_linear_tile_kernel<P, WM, WN, RA, RB, KS, DUAL>), dim3((unsigned)nbn * nbt * slabs), dim3(64 * S::NW * KS), S::LDS, st,
                     out, (const u16*)x, (const u16*)w, (const u16*)bias, T, N, K, epi, nbt, slabs, limit, alpha);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// ---- many tokens of a batch of small problems (per-head products): the same main loop, rows with strides of their own, 128 x 128 tiles of four
// waves, two workgroups a CU: K is a few stages, and one's stores run beside the other's products.  us, 64 x 64 tiles from L2 / this, bf16:
// 32 heads, fp32 out 512 x 128 at 128 / 400 / 1999 tokens 8.1 / 22.8 / 83 -> 5.9 / 9.1 / 29 (147 MB out), a gate per output 128 x 512 at
// 300 / 2048 19.7 / 64 -> 11.2 / 24; 16 heads 256 x 64 at 256 / 1101 5.7 / 15.9 -> 5.9 / 7.7, gated 64 x 256 at 700 / 2048 10.6 / 14.0 -> 9.5 / 9.9.  So from 96
// tiles on.
template <typename P>
__global__ __launch_bounds__(256, 2) void seq_linear_tile_batched_kernel(void* __restrict__ out_, const u16* __restrict__ x, const u16* __restrict__ w,
                                                                          int T, int N, int K, int epi, int nbt, int nbn, LinExt ext) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int WN = 2, RA = 4, RB = 4;
  typedef TileShape<2, WN, RA, RB, 1> S;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
  const int id = tile_of_block(blockIdx.x, gridDim.x), column = __builtin_amdgcn_readfirstlane(id / nbt), z = __builtin_amdgcn_readfirstlane(column / nbn);
  const int n0 = (column - z * nbn) * S::BN, t0 = (id - column * nbt) * S::BT;
  unsigned voff[S::NPW];
#pragma unroll
  for (int i = 0; i < S::NPW; ++i) {
    const int p = wave + S::NW * i;
    if (S::NW * i < S::NPA) voff[i] = tile_voff(p, lane, K, [&](int row) { return min(n0 + row, N - 1) - n0; });
    else voff[i] = tile_voff(p - S::NPA, lane, ext.ldx, [&](int row) { return min(t0 + row, T - 1) - t0; });
  }
  f32x4 acc[RA][RB];
  (void)tile_products<P, 2, WN, RA, RB, 1, false>(acc, smem, w + z * ext.sw + (long)n0 * K, x + z * ext.sx + (long)t0 * ext.ldx, 128, voff, K / 64, wave, 0);
  const int nw = n0 + wm * (16 * RA);
  const long obase = z * ext.so;
  const float* gate = ext.gate ? ext.gate + (long)z * ext.sg : nullptr;
  const unsigned strip = (unsigned)(size_t)(lds_char*)smem + (unsigned)wave * TileRows<16, RA>::BYTES;
  // the gates of all outputs are asked for at once, four (N % 4 == 0 here) or a row's one for all: fetched one by one in front of their quotients they were
  // four round trips of 16 loads, and up to a few hundred tiles the 64 x 64 ones were ahead (us, gate per output, those / one by one / at once: 16 x (256 x 64),
  // 300 tokens 9.8 / 14.0 / 8.5; 32 x (512 x 128), 128 tokens 11.6 / 14.8 / 9.2, 2048 168 / 82 / 49; 64 x (64 x 64), 256 tokens 9.5 / 13.7 / 8.5)
  typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
  f32x4 gv[RB][RA];
  if (gate) {
#pragma unroll
    for (int t = 0; t < RB; ++t) {
      const float* gr = gate + (long)min(t0 + (wn * RB + t) * 16 + j, T - 1) * ext.ldg;
#pragma unroll
      for (int i = 0; i < RA; ++i) {
        if (epi == EPI_GATE_ROW) gv[t][i] = i ? gv[t][0] : f32x4{gr[0], gr[0], gr[0], gr[0]};
        else gv[t][i] = *reinterpret_cast<const quad*>(gr + min(nw + i * 16 + 4 * g, N - 4));
      }
    }
  }
#pragma unroll
  for (int t = 0; t < RB; ++t) {
    const int tile0 = t0 + (wn * RB + t) * 16;
    f32x4 v[RA];
#pragma unroll
    for (int i = 0; i < RA; ++i) v[i] = acc[i][t];
    if (gate) {
#pragma unroll
      for (int i = 0; i < RA; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[i][r] = gated_(v[i][r], gv[t][i][r]);
    }
    if (epi == EPI_F32) {
      tile_rows_out<16, RA>(strip, v, [&](int row, int at, u32x4 b) {
        if (tile0 + row < T && nw + at / 4 < N) *reinterpret_cast<u32x4*>(reinterpret_cast<float*>(out_) + obase + (long)(tile0 + row) * ext.ldo + nw + at / 4) = b;
      });
      continue;
    }
    u32x2 d[RA];
#pragma unroll
    for (int i = 0; i < RA; ++i) d[i] = u32x2{pack2<P>(v[i][0], v[i][1]), pack2<P>(v[i][2], v[i][3])};
    tile_rows_out<8, RA>(strip, d, [&](int row, int at, u32x4 b) {
      if (tile0 + row < T && nw + at / 2 < N) *reinterpret_cast<u32x4*>(reinterpret_cast<u16*>(out_) + obase + (long)(tile0 + row) * ext.ldo + nw + at / 2) = b;
    });
  }
}

// whole 64-k stages, every row of every problem 16-byte aligned and stored in whole 16-byte groups, 32-bit offsets inside an operand
template <typename P>
static bool tile_batched_ok(const void* out, const void* x, const void* w, int T, int N, int K, int epi, const LinExt& ext, int batch) {
  if constexpr (sizeof(typename El<P>::type) == 4) return false;
  const int per = epi == EPI_F32 ? 4 : 8;                    // outputs of 16 bytes
  if ((long)((N + 127) / 128) * ((T + 127) / 128) * batch < 96) return false;
  return T >= 128 && N >= 64 && K % 64 == 0 && N % per == 0 && ext.ldo % per == 0 && ext.so % per == 0 && ext.ldx % 8 == 0 && ext.sx % 8 == 0 &&
         ext.sw % 8 == 0 && ((uintptr_t)out | (uintptr_t)x | (uintptr_t)w) % 16 == 0 && (long)ext.ldx * 256 < (1L << 31) && (N + 128L) * K < (1L << 31);
}
template <typename P>
static int launch_tile_batched(void* out, const void* x, const void* w, int T, int N, int K, int epi, const LinExt& ext, int batch, hipStream_t st) {
  typedef TileShape<2, 2, 4, 4, 1> S;
  if (ensure_dynamic_lds<seq_linear_tile_batched_kernel<P>>(S::LDS) != UMB_OK) return UMB_EHIP;
  const int nbn = (N + S::BN - 1) / S::BN, nbt = (T + S::BT - 1) / S::BT;
  if ((long)nbn * nbt * batch > 0x7fffffffL) return UMB_EINVAL;
  hipLaunchKernelGGL(seq_linear_tile_batched_kernel<P>, dim3((unsigned)nbn * nbt * batch), dim3(256), S::LDS, st, out, (const u16*)x, (const u16*)w, T, N, K,
                     epi, nbt, nbn, ext);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// us at T x N x K, two kinds of 256 x 256 / 128 x 128 tiles by a fixed share of a round (the rule before) -> tile_kind's: 1101 x 16384 x 2048 gate/up 109 -> 83,
// 2048 x 5120 x 2048 70 -> 48, 1101 x 2048 x 8192 79 -> 62, 2048 x 2048 x 2048 30 -> 22, 2466 x 4096 x 14336 376 -> 230, 700 x 4096 x 4096 47 -> 35, 512 x 2048 x 8192
// 73 -> 53; 2048 x 16384 x 2048 gate/up 126 -> 121 and 2048 x 28672 x 4096 412 -> 404 keep their tiles.
template <typename P, bool DUAL>
static int launch_tile(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, int slabs, float limit,
                       float alpha, hipStream_t st) {
  double us;
  const int kind = tile_kind(T, DUAL ? 2 * N : N, (K / 64 + slabs - 1) / slabs, slabs, K % (128 * slabs) == 0, &us);
  if (slabs == 1) {
    const TileMix mix = tile_mix(T, DUAL ? 2 * N : N, K / 64, us);
#define MIXED(KIND, RB) if (mix.columns && mix.tail == KIND) return launch_mixed<P, RB, DUAL>(out, x, w, bias, T, N, K, epi, mix.columns, limit, alpha, st)
    MIXED(TILE_192, 6);
    MIXED(TILE_160, 5);
    MIXED(TILE_128W, 4);
    MIXED(TILE_96, 3);
#undef MIXED
  }
  switch (kind) {
    case TILE_256: return launch_tile_as<P, 4, 2, 4, 8, 1, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
    case TILE_192: return launch_tile_as<P, 4, 2, 4, 6, 1, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
    case TILE_160: return launch_tile_as<P, 4, 2, 4, 5, 1, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
    case TILE_128W: return launch_tile_as<P, 4, 2, 4, 4, 1, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
    case TILE_96: return launch_tile_as<P, 4, 2, 4, 3, 1, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
    case TILE_128: return launch_tile_as<P, 2, 4, 4, 2, 1, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
    default: return launch_tile_as<P, 2, 2, 4, 2, 2, DUAL>(out, x, w, bias, T, N, K, epi, slabs, limit, alpha, st);
  }
}

// whole 64-k stages, 16-byte pieces and stores, 32-bit offsets inside an operand
static bool tile_ok(const void* out, const void* x, const void* w, int T, int N, int K, int epi) {
  const long rows = (epi_dual(epi) ? 2L : 1L) * N + 256;
  return K % 64 == 0 && rows * K < (1L << 31) && ((uintptr_t)out | (uintptr_t)x | (uintptr_t)w) % 16 == 0;
}

template <typename P>
static int launch_wide(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, hipStream_t st,
                       const LinExt& ext, int gy = 0) {
  if constexpr (sizeof(typename El<P>::type) == 2) {
    const unsigned ty = gy > 0 ? gy : (T + 127) / 128;
    if (epi_dual(epi))
      hipLaunchKernelGGL((seq_linear_wide_kernel<P, true>), dim3((N + 63) / 64, ty), dim3(256), 0, st, out,
                         (const u16*)x, (const u16*)w, (const u16*)bias, T, N, K, epi, ext);
    else
      hipLaunchKernelGGL((seq_linear_wide_kernel<P, false>), dim3((N + 127) / 128, ty), dim3(256), 0, st, out,
                         (const u16*)x, (const u16*)w, (const u16*)bias, T, N, K, epi, ext);
    UMB_LAUNCH_CHECK();
    return UMB_OK;
  } else {
    return UMB_EINVAL;
  }
}

// ---- whole 512-byte pieces of K: both operands of a step staged through LDS in contiguous runs.
// The kernel above asks for a fragment with one load of 16 rows x 64 B.  Rows of a power-of-two stride sit on the same L2 channel, so
// such a load takes ~75 cycles of a CU's path whether the rows are weights or tokens, and a launch of 16 and more tokens is bound by
// its TOKEN fragments (4096 x 14336 weights: 27 us with 1 token, 38 with 16, 80 with 64).  Here a workgroup walks K in chunks of 512
// bytes per row: LDS-DMA pieces of two rows (whole lines, 4 channels' worth each) into a ring of R slots, R - 1 chunks ahead, one
// barrier per chunk; the tokens of a chunk are fetched once per workgroup and not once per wave; fragments come from LDS without bank
// conflicts (pieces 1040 B apart, columns of odd rows XOR 8).  Wave w takes the 32-k steps w, w + 4, ... of a chunk.
// us, cold weights, one MI355X: 4096 x 14336, 1 / 16 / 48 / 64 tokens 27 / 38 / 66 / 80 -> 24 / 25 / 38 / 41; 2048 x 2048, 48 tokens
// 11.7 -> 7.3; gate/up 28672 x 4096, 1 / 16 / 48 tokens 49 / 58 / 88 -> 42 / 43 / 56 (5.6 TB/s at 1 token).
template <typename P, int NT, int TT, int BP, bool DUAL, int R, bool RUN>
__global__ __launch_bounds__(256) void seq_linear_stream_kernel(void* __restrict__ out_, const typename El<P>::type* __restrict__ x,
                                                                const typename El<P>::type* __restrict__ w,
                                                                const typename El<P>::type* __restrict__ bias, int T, int N, int K,
                                                                int epi, LinExt ext) {
  typedef typename El<P>::type E;
  typedef StreamShape<NT, TT, BP, DUAL, R> S;
  static_assert(S::rows_inside_slot(), "a fragment reads rows of the slot it belongs to and no others");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int EB = sizeof(E), STEPS = 512 / (32 * EB), AT = S::AT;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  int t0 = blockIdx.y * (TT * 16);
  const int ldx = ext.ldx, ldo = ext.ldo, parts = ext.parts, step = ext.step, turn = ext.turn;
  long obase = (long)blockIdx.z * ext.so;
  const float* gate = ext.gate ? ext.gate + (long)blockIdx.z * ext.sg : nullptr;
  x += (long)blockIdx.z * ext.sx;
  w += (long)blockIdx.z * ext.sw;
  if (ext.tiles) {                         // grouped: this workgroup's rows and weights come from the tile list
    const int* td = ext.tiles + 3 * blockIdx.y;
    const int rows = __builtin_amdgcn_readfirstlane(td[2]);
    if (rows <= 0) return;
    const long first = __builtin_amdgcn_readfirstlane(td[1]);
    w += (long)__builtin_amdgcn_readfirstlane(td[0]) * ext.gs;
    x += first * ldx;
    obase += first * ldo;
    T = rows;
    t0 = 0;
  }
  const unsigned lds0 = (unsigned)(size_t)(lds_char*)smem;
  // piece p: rows 2 p and 2 p + 1 (lanes 0 - 31, 32 - 63) of the operand; rows past its end re-read the last one: not stored
  unsigned voff[S::PW];
  auto rows_of_block = [&](int n0) {       // the weight pieces' offsets from row n0
#pragma unroll
    for (int i = 0; i < S::AP / 4; ++i) {
      const int odd = lane >> 5, c = (lane & 31) ^ (odd * 8), r = 2 * (wave + 4 * i) + odd;
      const int n = DUAL && r >= 16 * NT ? N + min(n0 + r - 16 * NT, N - 1) : min(n0 + r, N - 1);
      voff[i] = (unsigned)(n - n0) * (unsigned)K * EB + c * 16u;
    }
  };
#pragma unroll
  for (int i = S::AP / 4; i < S::PW; ++i) {
    const int odd = lane >> 5, c = (lane & 31) ^ (odd * 8);
    voff[i] = (unsigned)(min(t0 + 2 * (wave + 4 * i - S::AP) + odd, T - 1) - t0) * (unsigned)ldx * EB + c * 16u;
  }
  const char* wb = reinterpret_cast<const char*>(w);
  const char* xb = reinterpret_cast<const char*>(x + (long)t0 * ldx);
  int nc = K * EB / 512;
  if (parts > 1) {                         // this workgroup's slab of K: chunks c0 .. c0 + nc - 1
    const int z = blockIdx.z, longer = nc - parts * ext.part_chunks, c0 = z * ext.part_chunks + min(z, longer);
    nc = ext.part_chunks + (z < longer);
    wb += (long)c0 * 512;
    xb += (long)c0 * 512;
    if (z) bias = nullptr;
  }
  // the row blocks of this workgroup, blockIdx.x, + step, ...: their chunks are ONE sequence, the ring runs on over the end of a block
  const int nb = (N + 16 * NT - 1) / (16 * NT);
  int fb = blockIdx.x, left = nc;          // the block that is fetched, its chunks that are still to come
  int col = first_chunk(fb * (16 * NT), nc, turn);                // and the next of them: they are taken in turn from this one on
  const char* fw = wb + (long)fb * (16 * NT) * K * EB;
  rows_of_block(fb * (16 * NT));
  // Weights that one workgroup alone reads do not stay in L2: left there they push out the code, tokens, tables and partial sums of the dozen
  // small kernels around a product, each of which then fetched its own from further away (us, kept / not: one token, gate/up 28672 x 4096 41.9 / 41.1,
  // two-map attention 11.6 / 9.7, delta rule 10.2 / 8.4; a whole call of 17 steps, 8B widths, 16 requests 8936 / 8531, one 7290 / 6824).  From 33 tokens
  // on the tokens' own pieces are more than the weights, and 48 tokens of 1B widths were 2 % slower for it.  Tile lists: two tiles may share weights.
  const bool once = TT <= 2 && !ext.tiles;
  auto issue = [&](int slot) {
    const long at = (long)col * 512;
    col = col + 1 == nc ? 0 : col + 1;     // past the last chunk of all: fetched again, never read
    --left;
#pragma unroll
    for (int i = 0; i < S::PW; ++i) {
      unsigned dst = lds0 + (unsigned)slot * S::SLOT + (unsigned)(wave + 4 * i) * S::PIECE;
      if (S::NP % 4 && i == S::PW - 1 && wave + 4 * i >= S::NP) dst = lds0 + (unsigned)R * S::SLOT;      // a piece of nobody's
      if (4 * i >= S::AP) tile_dma(voff[i], xb + at, dst);
      else if (once) tile_dma_once(voff[i], fw + at, dst);
      else tile_dma(voff[i], fw + at, dst);
    }
  };
  f32x4 acc[AT][TT];
#pragma unroll
  for (int i = 0; i < AT; ++i)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[i][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned wrow = S::weight_row(0, j), trow = S::token_row(0, j), swz = (unsigned)(j & 1) * 8u;
  auto frag = [&](unsigned base, int s) {  // this lane's part of 16 rows, the 32 k of step s
    const auto at = [&](int c) { return *reinterpret_cast<const lds_u32x4*>((size_t)(base + (((unsigned)c) ^ swz) * 16u)); };
    Frag8<P> f;
    if constexpr (EB == 2) f.v = at(s * 4 + g);
    else {
      f.lo = __builtin_bit_cast(f32x4, at(s * 8 + 2 * g));
      f.hi = __builtin_bit_cast(f32x4, at(s * 8 + 2 * g + 1));
    }
    return f;
  };
#pragma unroll
  for (int c = 0; c < R - 1; ++c) issue(c);
  int slot = 0;
  for (int block = blockIdx.x; block < nb; block += step) {
    const int n0 = block * 16 * NT;
#pragma unroll
    for (int i = 0; i < AT; ++i)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) acc[i][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    unsigned base = lds0;
    for (int c = 0; c < nc; ++c) {
      // this wave's pieces of the chunk have landed and its fragments of the chunk before are in registers; behind the barrier that holds
      // for every wave: the chunk can be read, and the slot of the chunk before filled again
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((R - 2) * S::PW) : "memory");
      __builtin_amdgcn_s_barrier();
      if (RUN && __builtin_expect(left == 0 && fb + step < nb, 0)) {
        fb += step;
        left = nc;
        col = first_chunk(fb * (16 * NT), nc, turn);
        fw = wb + (long)fb * (16 * NT) * K * EB;
        rows_of_block(fb * (16 * NT));
      }
      issue(slot == 0 ? R - 1 : slot - 1);
      base = lds0 + (unsigned)slot * S::SLOT;
#pragma unroll
      for (int u = 0; u < STEPS / 4; ++u) {
        const int s = wave + 4 * u;
        Frag8<P> a[AT], b[TT];
#pragma unroll
        for (int i = 0; i < AT; ++i) a[i] = frag(base + wrow + (unsigned)(8 * i) * S::PIECE, s);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) b[tt] = frag(base + trow + (unsigned)(8 * tt) * S::PIECE, s);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
          for (int i = 0; i < AT; ++i) acc[i][tt] = mma8<P>(a[i], b[tt], acc[i][tt]);
      }
      slot = slot + 1 == R ? 0 : slot + 1;
    }
    // the waves' tiles are added in the slot of the block's last chunk, which the next block's first barrier hands back to the ring; behind the
    // last block nothing of this wave may be writing LDS any more (waited for here, not behind the stores: those need no wait)
    if (!RUN || block + step >= nb) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const unsigned red = base;                                         // [wave][AT][TT][256] floats
#pragma unroll
    for (int i = 0; i < AT; ++i)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) *reinterpret_cast<lds_f32x4*>((size_t)(red + (((wave * AT + i) * TT + tt) * 256 + lane * 4) * 4u)) = acc[i][tt];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const int l = threadIdx.x >> 2, r = threadIdx.x & 3;
    auto total = [&](int i, int tt) {
      const auto at = [&](int ww) { return *reinterpret_cast<const lds_f32*>((size_t)(red + (((ww * AT + i) * TT + tt) * 256 + threadIdx.x) * 4u)); };
      float s = at(0);
#pragma unroll
      for (int ww = 1; ww < 4; ++ww) s += at(ww);
      return s;
    };
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = n0 + nt * 16 + 4 * (l >> 4) + r;
      if (n >= N) continue;
      const float bv = bias ? ldf<P>(bias + n) : 0.f;
      const float bv2 = (DUAL && bias) ? ldf<P>(bias + N + n) : 0.f;
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const int t = t0 + tt * 16 + (l & 15);
        if (t >= T) continue;
        const float s = total(nt, tt) + bv;
        const long o = obase + (long)t * ldo + n;
        if constexpr (DUAL) {
          stf<P>(reinterpret_cast<E*>(out_) + o, glu_pair(epi, s, total(NT + nt, tt) + bv2, ext.limit, ext.alpha));
        } else if (epi == EPI_DT) {
          stf<P>(reinterpret_cast<E*>(out_) + o, s);
        } else if (epi == EPI_RELU2) {
          const float rl = fmaxf(s, 0.f);
          stf<P>(reinterpret_cast<E*>(out_) + o, rl * rl);
        } else if (epi == EPI_GATE) {
          stf<P>(reinterpret_cast<E*>(out_) + o, s / (1.f + expf(-gate[(long)t * ext.ldg + n])));
        } else if (epi == EPI_GATE_ROW) {
          stf<P>(reinterpret_cast<E*>(out_) + o, s / (1.f + expf(-gate[(long)t * ext.ldg])));
        } else if (epi == EPI_CAP) {
          reinterpret_cast<float*>(out_)[o] = ext.limit * tanhf(s / ext.limit);
        } else {
          reinterpret_cast<float*>(out_)[o] = s;
        }
      }
    }
    if (!RUN) break;
  }
}

template <typename P, int NT, int TT, int BP, bool DUAL, int R, bool RUN>
static int launch_stream_grid(dim3 grid, void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, hipStream_t st,
                              LinExt ext) {
  typedef typename El<P>::type E;
  typedef StreamShape<NT, TT, BP, DUAL, R> S;
  if (ensure_dynamic_lds<seq_linear_stream_kernel<P, NT, TT, BP, DUAL, R, RUN>>(S::LDS) != UMB_OK) return UMB_EHIP;
  ext.step = (int)grid.x;
  hipLaunchKernelGGL((seq_linear_stream_kernel<P, NT, TT, BP, DUAL, R, RUN>), grid, dim3(256), S::LDS, st, out, (const E*)x, (const E*)w, (const E*)bias,
                     T, N, K, epi, ext);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
// Workgroups, and row blocks for each.  held > 0: so many workgroups at most, each running on from block to block, the ring filled across their ends (a new
// workgroup's first chunks and its last sums would stand bare); 0: a block each.
template <typename P, int NT, int TT, int BP, bool DUAL, int R, bool RUN>
static int launch_stream_as(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, hipStream_t st,
                            LinExt ext, int gy, int gz, int held) {
  const long chunks = (long)K * sizeof(typename El<P>::type) / 512;
  ext.turn = chunks >= 8 && gy == 0 && (gz == 1 || ext.parts > 1) ? 7 : 0;
  const int blocks = (N + 16 * NT - 1) / (16 * NT), ty = gy > 0 ? gy : (T + 16 * TT - 1) / (16 * TT);
  if constexpr (RUN)
    if (ty == 1 && gz == 1 && blocks > held && chunks >= R)
      return launch_stream_grid<P, NT, TT, BP, DUAL, R, true>(dim3(held), out, x, w, bias, T, N, K, epi, st, ext);
  return launch_stream_grid<P, NT, TT, BP, DUAL, R, false>(dim3(blocks, ty, gz), out, x, w, bias, T, N, K, epi, st, ext);
}

// workgroups that run on: two a unit, or one where whole rounds of two would do more than a tenth beyond the blocks that there are
static inline int stream_held(long blocks) { return 10 * ((blocks + 511) / 512 * 512) > 11 * ((blocks + 255) / 256 * 256) ? 256 : 512; }

// T: tokens of a token tile at most (grouped launches), of the launch otherwise.  32 output rows a workgroup halve the token traffic of launches that
// stay above one workgroup per CU (32000 x 2048, 48 tokens 51 -> 37 us; 4096 x 4096, 256 workgroups of 16 rows: 12.4 us, 15.3 as 128 of 32).
// How many chunks ahead: a unit streams best with some 30 to 60 KB under way, its tokens' among them, however many workgroups share it -- fewer leave it
// waiting, more are slower by a tenth (the memory serves rows of 512 bytes from too many places).  So a ring of four slots where a unit has one workgroup,
// of three for two, of two for more, and a launch of more blocks than that runs on inside one or two workgroups a unit.  us, bf16, cold weights, one MI355X,
// four (gate and up: three; 32 tokens three and two) slots whatever the launch / this:
//   1 token   6144 x 4096 10.9 / 10.2, 12304 x 4096 19.5 / 16.7, 12304 x 2048 12.4 / 9.9, 32000 x 2048 23.0 / 21.9, gate/up 14336 x 4096 40.4 / 37.5, 8192 x 2048 13.9 / 12.9
//   16        8192 x 4096 14.6 / 13.5, 12304 x 4096 22.7 / 20.5, 10304 x 4096 19.7 / 16.5, gate/up 14336 x 4096 40.6 / 38.4, 28672 x 4096 73 / 68
//   32        6144 x 4096 16.9 / 13.7, 12304 x 4096 29.1 / 23.4, 32000 x 2048 33.2 / 26.0, gate/up 11008 x 4096 42.1 / 34.2
template <typename P>
static int launch_stream(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, hipStream_t st,
                         const LinExt& ext, int gy = 0, int gz = 1) {
#define STREAM(NT, TT, BP, DUAL, R, RUN, HELD) return launch_stream_as<P, NT, TT, BP, DUAL, R, RUN>(out, x, w, bias, T, N, K, epi, st, ext, gy, gz, HELD)
  const long blocks = (long)((N + 15) / 16) * gz, chunks = (long)K * sizeof(typename El<P>::type) / 512;
  // true fp32 of more than 8 tokens stands on its products: as many waves on a unit as before
  constexpr bool F = sizeof(typename El<P>::type) == 4;
  if constexpr (!F)
    if (gy == 0 && gz == 1 && ext.parts <= 1 && !ext.tiles && ext.ldx == K && ext.ldo == N && held_pays(T, N, K, epi))
      return held_stream(out, x, w, bias, T, N, K, epi, ext.limit, ext.alpha, std::is_same<P, BF16>::value ? UMB_SEQ_BF16 : UMB_SEQ_F16, st);
  if (epi_dual(epi)) {
    // up to some 1.5 blocks a unit they stand side by side: a second one behind the first would leave half of the units idle (fp32: 1.75; 6912 x 1024 of
    // one token side by side / behind one another 12.3 / 12.9, 8192 14.0 / 13.6)
    const int held = blocks <= (F ? 448 : 400) ? 512 : 256;
    // fp32 of more than 12 chunks: a workgroup a block, two on a unit -- one alone is too few waves for its products (us, one block behind the other / this: 2 tokens,
    // 12320 x 1792 41.4 / 36.0, 5 tokens, 15328 x 1792 43.7 / 40.2; over 3000 launches of 450 to 2048 blocks 1 % behind to 5 % ahead in the median of a size)
    if (F && chunks > 12 && T <= 8) STREAM(1, 1, 4, true, 3, false, 0);
    if (T <= 8) STREAM(1, 1, 4, true, 3, true, held);
    if (T <= 16) STREAM(1, 1, 8, true, 3, true, F ? 1 << 30 : held);
    if (T <= 32) {
      // (two blocks a unit stand side by side: 17 tokens, 6864 x 2816 18.3 us, 19.7 behind one another; 1 to 2 % in the median of 8000 launches)
      if (F || chunks < 3 || (blocks > 256 && blocks <= 512)) STREAM(1, 2, 16, true, 2, false, 0);
      STREAM(1, 2, 16, true, 3, true, 256);
    }
    if (T <= 48) STREAM(1, 3, 24, true, 3, true, 256);
    STREAM(1, 4, 32, true, 3, true, 256);
  }
  if (T <= 8) {
    if (gy > 0 || blocks <= 256) STREAM(1, 1, 4, false, 4, false, 0);
    if (blocks <= 512) STREAM(1, 1, 4, false, 3, false, 0);
    if (blocks <= 1024 || gz > 1) STREAM(1, 1, 4, false, 2, false, 0);
    if constexpr (F) STREAM(1, 1, 4, false, 4, true, 768);
    if (stream_held(blocks) == 512) STREAM(1, 1, 4, false, 3, true, 512);
    STREAM(1, 1, 4, false, 4, true, 256);
  }
  if (T <= 16) {
    if (F) STREAM(1, 1, 8, false, 4, true, 512);
    if (gy > 0 || blocks <= 256) STREAM(1, 1, 8, false, 4, false, 0);
    if (gz > 1 && blocks <= 512) STREAM(1, 1, 8, false, 3, false, 0);
    if (gz > 1 || (blocks > 512 && blocks <= 1024)) STREAM(1, 1, 8, false, 2, false, 0);
    STREAM(1, 1, 8, false, 4, true, 256);
  }
  const bool narrow = stream_narrow(N, gy > 0 ? (gy + 1) / 2 : (T + 63) / 64, gz);    // about half of a tile list is in use
  if (T <= 32) {
    if (narrow) STREAM(1, 2, 16, false, 3, false, 0);
    // (K of two chunks cannot run on in a ring of three: 24 tokens, 16400 x 512 10.7 / 7.7, 50000 x 512 26.6 / 15.8)
    if (blocks <= 512 || (!F && chunks >= 3 && stream_held((blocks + 1) / 2) == 256)) STREAM(2, 2, 16, false, 3, true, 256);
    // (fp32 whose blocks of 32 rows are a few more than two a unit holds: three rounds of 16 rows are less than two of 32; 17 tokens, 18768 x 2816 55.5 / 51.8 us,
    // 2 to 5 % in the median of 8000 launches)
    if (F && chunks > 2 && blocks > 1024 && blocks <= 1280) STREAM(1, 2, 16, false, 3, true, 512);
    STREAM(2, 2, 16, false, 2, true, 512);
  }
  if (T <= 48) {
    if (narrow) STREAM(1, 3, 24, false, 3, false, 0);
    STREAM(2, 3, 24, false, 3, true, 256);
  }
  if (narrow) STREAM(1, 4, 32, false, 3, false, 0);
  STREAM(2, 4, 32, false, 3, true, 256);
#undef STREAM
}

// The same for tile lists, whose tiles in use are not known here (bf16, eight experts, two a token; us, one-tile kernel / ring): tiles of
// 16 rows, single matrices: 2048 x 2048 12.7 / 14.5 at 4 tokens, 4096 x 1024 15.2 / 18.7 at 16, 4096 x 3584 47 / 43, 1024 x 2048 8.8 / 8.4;
// gate and up together 28672 x 4096 94 / 81.  Tiles of 64 rows: 4096 x 1024 17.5 / 23.3 at 64 tokens, gate and up 8192 x 2048 37 / 38, 3584 x 4096
// 56 / 62 at 33; 1024 x 1024 12 / 7.3; fp32 2048 x 512 16.6 / 18.2 at 33, 2048 x 2048 67 / 54.
static bool stream_pays_grouped(int tile_rows, int N, int K, int epi, int eb) {
  const long chunks = (long)K * eb / 512;
  const bool dual = epi_dual(epi);
  if (eb == 4) return tile_rows == 16 || chunks >= 16 || (dual ? 2 : 1) * N <= 128 * chunks;
  if (tile_rows == 16) return dual || chunks >= 12 || N <= 128 * chunks;
  return dual ? chunks >= 12 || 2 * N <= 384 * chunks : N <= 384 * chunks && N < 3584;
}

// gy > 0: the number of token tiles is given (grouped launches); gz: independent problems
template <typename P, int NT, int TT, bool VEC>
static int launch_tt(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, hipStream_t st,
                     const LinExt& ext, int gy = 0, int gz = 1) {
  typedef typename El<P>::type E;
  constexpr int NTD = NT > 2 ? 2 : NT;             // gate/up: two tile pairs at most
  const dim3 grid((N + NT * 16 - 1) / (NT * 16), gy > 0 ? gy : (T + TT * 16 - 1) / (TT * 16), gz);
  if (epi_dual(epi))
    hipLaunchKernelGGL((seq_linear_kernel<P, NTD, TT, VEC, true>), dim3((N + NTD * 16 - 1) / (NTD * 16), grid.y, gz), dim3(256), 0,
                       st, out, (const E*)x, (const E*)w, (const E*)bias, T, N, K, epi, ext);
  else
    hipLaunchKernelGGL((seq_linear_kernel<P, NT, TT, VEC, false>), grid, dim3(256), 0, st, out, (const E*)x, (const E*)w,
                       (const E*)bias, T, N, K, epi, ext);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// Whether a dense product of more than 64 tokens takes the staged tiles (stream: the streaming kernel takes it otherwise).  Both operands are
// re-used: from 256 tokens on, and for 65 and more where the launch has some 100 tiles of 128 x 128 (cold weights, 100 / 200 tokens: 18496 x 4096
// 56 / 72 us, the streaming kernel 84 / 158; 4096 x 4096 41 / 39 us, streaming 18 / 32; 2048 x 8192, 255 tokens 73 us, streaming 29)
static bool tiles_pay(int T, long rows, bool stream) {
  const long tiles = (rows + 127) / 128 * ((T + 127) / 128);
  return !(stream && tiles < (T < 256 ? 96 : 49)) && (T >= 256 || tiles >= 96);
}

template <typename P, bool VEC>
static int launch_vec(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, hipStream_t st,
                      const LinExt& ext, int gz = 1) {
  const bool dense = gz == 1 && ext.ldx == K && ext.ldo == N && epi != EPI_GATE && epi != EPI_GATE_ROW;
  constexpr int EB = sizeof(typename El<P>::type);
  const bool stream = VEC && stream_ok(x, w, N, K, epi, ext, EB) && stream_pays(T, N, K, epi, gz, EB);
  if constexpr (sizeof(typename El<P>::type) == 2) {
    if (T > 64 && VEC && dense && N >= 128 && tile_ok(out, x, w, T, N, K, epi) && tiles_pay(T, (long)(epi_dual(epi) ? 2 : 1) * N, stream))
      return epi_dual(epi) ? launch_tile<P, true>(out, x, w, bias, T, N, K, epi, 1, ext.limit, ext.alpha, st)
                           : launch_tile<P, false>(out, x, w, bias, T, N, K, epi, 1, ext.limit, ext.alpha, st);
  }
  if (stream) return launch_stream<P>(out, x, w, bias, T, N, K, epi, st, ext, 0, gz);
  if (T <= 16) return launch_tt<P, 1, 1, VEC>(out, x, w, bias, T, N, K, epi, st, ext, 0, gz);
  if (T <= 32) return launch_tt<P, 1, 2, VEC>(out, x, w, bias, T, N, K, epi, st, ext, 0, gz);
  // many tokens: the launch is bound by fragment loads per MFMA, not by weight bytes -> four output tiles per workgroup
  // (the K order of every output is unchanged)
  if (T > 64 && N >= 64 && sizeof(typename El<P>::type) == 2) {
    if (VEC && dense && T >= 256 && N >= 128) return launch_wide<P>(out, x, w, bias, T, N, K, epi, st, ext);      // both operands re-used
    return launch_tt<P, 4, 4, VEC>(out, x, w, bias, T, N, K, epi, st, ext, 0, gz);
  }
  return launch_tt<P, 1, 4, VEC>(out, x, w, bias, T, N, K, epi, st, ext, 0, gz);
}

static int seq_linear_any(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, float limit,
                          float alpha, int dtype, hipStream_t st) {
  if (T < 1 || N < 1 || K < 1 || !(epi_plain(epi) || epi == EPI_CLAMP_GLU || epi == EPI_CAP) || !out || !x || !w) return UMB_EINVAL;
  if (epi_dual(epi)) {
    if (N & 1) return UMB_EINVAL;
    N >>= 1;                                   // rows of each half
  }
  LinExt ext = lin_dense(N, K);
  ext.limit = limit;
  ext.alpha = alpha;
  DISPATCH_SEQ_DTYPE(dtype, {
    if (K % 8 == 0) return launch_vec<P, true>(out, x, w, bias, T, N, K, epi, st, ext);
    return launch_vec<P, false>(out, x, w, bias, T, N, K, epi, st, ext);
  })
}

extern "C" int umb_seq_linear(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, int dtype,
                              hipStream_t st) {
  if (!epi_plain(epi)) return UMB_EINVAL;                   // the others have constants: umb_seq_linear_glu, umb_seq_linear_cap
  return seq_linear_any(out, x, w, bias, T, N, K, epi, 0.f, 0.f, dtype, st);
}

// Slabs of K for a product whose partial sums the kernel behind it adds (the seams), 1: none.  Up to 64 tokens their number follows from the weights
// alone, so a token's sums are the same whatever else is in its step.  One workgroup per 16 output rows leaves half of the compute units idle below
// 128 of them, and from 33 tokens on a unit's path is full of token pieces that slabs with 32 output rows each halve; a slab is four chunks at
// least (shorter ones are all prologue).  us at 1 / 16 / 48 tokens, bf16, cold weights, one MI355X, 1 slab -> this rule's: 2048 x 8192 10.5 / 12.1 / 18.9 ->
// 8.8 / 9.5 / 10.8 (4); 2048 x 2048 4.6 / 5.0 / 7.2 -> 3.9 / 4.1 / 5.4 (2); 2560 x 6912 9.3 / 11.1 / 15.3 -> 8.3 / 9.9 / 10.6 (3).  Two slabs of more than 128
// workgroups are behind up to 32 tokens and ahead beyond (with the seam behind it, 1 / 16 / 32 / 48 tokens, 1 -> 2: 4096 x 14336 27.3 / 27.7 / 33.6 /
// 41.3 -> 28.0 / 29.2 / 35.6 / 31.7, 4096 x 4096 11.4 / 12.4 / 14.3 / 16.4 -> 12.0 / 13.3 / 15.2 / 14.9, 4096 x 8192 18.6 / 17.9 / 21.0 / 24.7 -> 21.6 / 20.8 /
// 23.1 / 22.5): K whole, for decoding of small batches.
//
// Many tokens: the staged tiles, where rounds of them fill better with K in slabs than the whole K does: the least of the product's time and of
// reading the slabs beyond the first in the kernel behind it (8 TB/s, they come from the last-level cache), against the whole K on the tiles or on
// the streaming kernel (0.50 us a chunk and round of 16 rows x 64 tokens a workgroup, 0.78 of 32).  us, whole / this: 4096 x 14336 at 100 / 300 / 1101 /
// 1999 tokens 46 / 95 / 171 / 198 -> 33 / 52 / 121 / 178; 2048 x 8192 at 128 / 300 / 1101 20.9 / 47 / 62 -> 20.9 / 22 / 42; 4096 x 4096 at 1101 53 -> 42.
// Their number follows from the tokens and the weights and not from the room that a caller happens to have: at most SLAB_ROWS rows of partial sums.
constexpr int SLAB_ROWS = 8192;
static int tile_slabs(int T, int N, int K, bool stream) {
  double best = 1e30, us = 0.0;
  if (tiles_pay(T, N, stream)) {
    (void)tile_kind(T, N, K / 64, 1, K % 128 == 0, &best);
  } else if (stream) {
    const bool narrow = stream_narrow(N, (T + 63) / 64, 1);
    const long wgs = (long)((N + (narrow ? 15 : 31)) / (narrow ? 16 : 32)) * ((T + 63) / 64);
    best = 2.5 + (wgs + 255) / 256 * (K / 256) * (narrow ? 0.50 : 0.78);
  }
  int best_s = 1;
  for (int S = 2; S <= 4 && S * 4 <= K / 64 && S <= SLAB_ROWS / T; ++S) {
    (void)tile_kind(T, N, (K / 64 + S - 1) / S, S, K % (128 * S) == 0, &us);
    us += (S - 1) * (double)T * N * 4 / 8e6;
    if (us < best) { best = us; best_s = S; }
  }
  return best_s;
}

extern "C" int umb_seq_tile_kind(int T, int rows, int K, int slabs) {
  if (T < 1 || rows < 1 || K < 64 || slabs < 1) return UMB_EINVAL;
  return tile_kind(T, rows, (K / 64 + slabs - 1) / slabs, slabs, K % (128 * slabs) == 0);
}

extern "C" int umb_seq_tile_mix(int T, int rows, int K) {
  if (T < 1 || rows < 1 || K < 64) return UMB_EINVAL;
  double us;
  (void)tile_kind(T, rows, K / 64, 1, K % 128 == 0, &us);
  const TileMix mix = tile_mix(T, rows, K / 64, us);
  return mix.columns * TILE_288 + mix.tail;              // (TILE_288 is none of this library's)
}

extern "C" int umb_seq_linear_split(const void* x, const void* w, int T, int N, int K, int dtype) {
  if (T < 1 || N < 1 || K < 1) return 1;
  const int eb = (int)seq_elem_bytes(dtype), chunks = (int)((long)K * eb / 512), blocks = (N + 15) / 16;
  const bool stream = stream_ok(x, w, N, K, EPI_F32, lin_dense(N, K), eb);
  if (T > 64) return eb == 2 && N >= 128 && tile_ok(nullptr, x, w, T, N, K, EPI_F32) ? tile_slabs(T, N, K, stream && stream_pays(T, N, K, EPI_F32, 1, eb)) : 1;
  if (!stream) return 1;
  const int parts = std::min(std::min(512 / blocks, 4), chunks / 4);
  return parts < 2 || (parts == 2 && blocks > 128) ? 1 : parts;
}

extern "C" int umb_seq_linear_parts(float* out, const void* x, const void* w, const void* bias, int T, int N, int K, int parts, int dtype,
                                    hipStream_t st) {
  if (T < 1 || N < 1 || K < 1 || parts < 1 || !out || !x || !w) return UMB_EINVAL;
  if (parts == 1) return umb_seq_linear(out, x, w, bias, T, N, K, EPI_F32, dtype, st);
  LinExt ext = lin_dense(N, K);
  ext.so = (long)T * N;
  ext.parts = parts;
  ext.part_chunks = (int)((long)K * seq_elem_bytes(dtype) / 512) / parts;
  if (T > 64) {
    if (parts > K / 64 || !tile_ok(out, x, w, T, N, K, EPI_F32)) return UMB_EINVAL;
    if (dtype == UMB_SEQ_BF16) return launch_tile<BF16, false>(out, x, w, bias, T, N, K, EPI_F32, parts, 0.f, 0.f, st);
    if (dtype == UMB_SEQ_F16) return launch_tile<F16, false>(out, x, w, bias, T, N, K, EPI_F32, parts, 0.f, 0.f, st);
    return UMB_EINVAL;
  }
  DISPATCH_SEQ_DTYPE(dtype, {
    constexpr int EB = sizeof(typename El<P>::type);
    if (parts > (long)K * EB / 512 || !stream_ok(x, w, N, K, EPI_F32, ext, EB)) return UMB_EINVAL;
    return launch_stream<P>(out, x, w, bias, T, N, K, EPI_F32, st, ext, 0, parts);
  })
}

extern "C" int umb_seq_linear_glu(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, float limit,
                                  float alpha, int dtype, hipStream_t st) {
  if (!(limit > 0.f)) return UMB_EINVAL;
  return seq_linear_any(out, x, w, bias, T, N, K, EPI_CLAMP_GLU, limit, alpha, dtype, st);
}

extern "C" int umb_seq_linear_cap(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, float cap, int dtype,
                                  hipStream_t st) {
  if (!(cap > 0.f)) return UMB_EINVAL;
  return seq_linear_any(out, x, w, bias, T, N, K, EPI_CAP, cap, 0.f, dtype, st);
}

extern "C" int umb_seq_linear_batched(void* out, const void* x, const void* w, int T, int N, int K, int ldx, int ldo, int batch,
                                      long sx, long sw, long so, int epi, const float* gate, int ldg, int sg, int dtype,
                                      hipStream_t st) {
  if (T < 1 || N < 1 || K < 1 || batch < 1 || batch > 65535 || ldx < K || ldo < N || !out || !x || !w ||
      !(epi == EPI_F32 || epi == EPI_DT || epi == EPI_GATE || epi == EPI_GATE_ROW) || ((epi == EPI_GATE || epi == EPI_GATE_ROW) && !gate))
    return UMB_EINVAL;
  const LinExt ext{ldx, ldo, 0, 0, 0, 0, sx, sw, so, 0, nullptr, gate, ldg, sg, 0.f, 0.f};
  // 16-byte loads need every row start aligned: the strides as well as K
  const bool vec = K % 8 == 0 && ldx % 8 == 0 && sx % 8 == 0 && sw % 8 == 0;
  DISPATCH_SEQ_DTYPE(dtype, {
    if constexpr (sizeof(typename El<P>::type) == 2)
      if (tile_batched_ok<P>(out, x, w, T, N, K, epi, ext, batch)) return launch_tile_batched<P>(out, x, w, T, N, K, epi, ext, batch, st);
    if (vec) return launch_vec<P, true>(out, x, w, nullptr, T, N, K, epi, st, ext, batch);
    return launch_vec<P, false>(out, x, w, nullptr, T, N, K, epi, st, ext, batch);
  })
}

static int seq_linear_grouped_any(void* out, const void* x, const void* w, const int* tiles, int max_tiles, int tile_rows, long gs,
                                  int N, int K, int epi, float limit, float alpha, int dtype, hipStream_t st) {
  if (max_tiles < 1 || max_tiles > 65535 || N < 1 || K < 1 || !(epi_plain(epi) || epi == EPI_CLAMP_GLU) || !out ||
      !x || !w || !tiles ||
      (tile_rows != 16 && tile_rows != 64 && tile_rows != 128))
    return UMB_EINVAL;
  if (epi_dual(epi)) {
    if (N & 1) return UMB_EINVAL;
    N >>= 1;
  }
  const LinExt ext{K, N, 0, 0, 0, 0, 0, 0, 0, gs, tiles, nullptr, 0, 0, limit, alpha};
  if (tile_rows == 128) {                  // many rows per group: both operands staged through LDS (16-bit storage only)
    if (dtype == UMB_SEQ_F32 || K % 8 || gs % 8) return UMB_EINVAL;
    if (dtype == UMB_SEQ_BF16) return launch_wide<BF16>(out, x, w, nullptr, 128, N, K, epi, st, ext, max_tiles);
    return launch_wide<F16>(out, x, w, nullptr, 128, N, K, epi, st, ext, max_tiles);
  }
  if (tile_rows == 16) {                   // a few rows in all (decoding): one 16-row output tile per workgroup, many workgroups
    DISPATCH_SEQ_DTYPE(dtype, {
      constexpr int EB = sizeof(typename El<P>::type);
      if (stream_ok(x, w, N, K, epi, ext, EB) && stream_pays_grouped(16, N, K, epi, EB)) return launch_stream<P>(out, x, w, nullptr, 16, N, K, epi, st, ext, max_tiles);
      if (K % 8 == 0 && gs % 8 == 0) return launch_tt<P, 1, 1, true>(out, x, w, nullptr, 16, N, K, epi, st, ext, max_tiles);
      return launch_tt<P, 1, 1, false>(out, x, w, nullptr, 16, N, K, epi, st, ext, max_tiles);
    })
  }
  DISPATCH_SEQ_DTYPE(dtype, {
    constexpr int EB = sizeof(typename El<P>::type);
    if (stream_ok(x, w, N, K, epi, ext, EB) && stream_pays_grouped(64, N, K, epi, EB)) return launch_stream<P>(out, x, w, nullptr, 64, N, K, epi, st, ext, max_tiles);
    if (K % 8 == 0 && gs % 8 == 0) {
      if (N >= 64 && sizeof(typename El<P>::type) == 2) return launch_tt<P, 4, 4, true>(out, x, w, nullptr, 64, N, K, epi, st, ext, max_tiles);
      return launch_tt<P, 1, 4, true>(out, x, w, nullptr, 64, N, K, epi, st, ext, max_tiles);
    }
    return launch_tt<P, 1, 4, false>(out, x, w, nullptr, 64, N, K, epi, st, ext, max_tiles);
  })
}

extern "C" int umb_seq_linear_grouped(void* out, const void* x, const void* w, const int* tiles, int max_tiles, int tile_rows,
                                      long gs, int N, int K, int epi, int dtype, hipStream_t st) {
  if (!epi_plain(epi)) return UMB_EINVAL;
  return seq_linear_grouped_any(out, x, w, tiles, max_tiles, tile_rows, gs, N, K, epi, 0.f, 0.f, dtype, st);
}

extern "C" int umb_seq_linear_grouped_glu(void* out, const void* x, const void* w, const int* tiles, int max_tiles, int tile_rows,
                                          long gs, int N, int K, float limit, float alpha, int dtype, hipStream_t st) {
  if (!(limit > 0.f)) return UMB_EINVAL;
  return seq_linear_grouped_any(out, x, w, tiles, max_tiles, tile_rows, gs, N, K, EPI_CLAMP_GLU, limit, alpha, dtype, st);
}
