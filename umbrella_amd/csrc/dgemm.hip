// Wide verify / prompt GEMM of dense 16-bit weights:  out[t][n] = sum_k x[t][k] * W[n][k],  T > 64 tokens, weights in gemm.hip's tile order.
//
// Reference call sites: the nn.Linear products of umbrella/models/llama.py (layer_compute, 75-134) at prompts and wide trees.
//
// Matrix-pipe bound.  The main loop is that of gemm_tile.h; the packed weights are MFMA fragments already, so a 1-KiB LDS-DMA piece of A
// is one fragment.  The register-resident kernel it replaces (gemm.hip: 64 x 128 per wave, activations staged through registers, two
// barriers a step) reached 610 - 730 TFLOP/s on 8B shapes at 1024 tokens; this one 900 - 1200 (figures: dgemm_tile).
// Split-K partials and epilogues are those of gemm.hip (fp32 [S][T][N]; rounded fp32; SiLU(gate) * up of interleaved rows, S = 1).
#include "gemm_fused.h"
#include "gemm_tile.h"
#include <cstdlib>

// A workgroup of the launch: tile number `tile` of nbt token tiles a column, slab sp of S, the columns from row `first` on.
template <typename P, int WM, int WN, int RA, int RB, int KS>
__device__ __forceinline__ void dgemm_block(unsigned char* smem, const unsigned char* __restrict__ wp, const u16* __restrict__ x, int ldx, int T, int N, int K,
                                            int S, int epi, int nbt, float* __restrict__ out, const GemmFused& fx, int tile, int sp, int first) {
  typedef TileShape<WM, WN, RA, RB, KS> Sh;
  const int lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_all % Sh::NW, ks = wave_all / Sh::NW, j = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
  const int n0 = first + (tile / nbt) * Sh::BN, t0 = (tile % nbt) * Sh::BT;
  const int nst = K / 64, per = (nst + S - 1) / S, st0 = min(nst, sp * per), st1 = min(nst, st0 + per);
  const int last = (N - n0) / 16 - 1;                        // row tiles and rows past the operand's end re-read its last one: not stored
  unsigned voff[Sh::NPW];
#pragma unroll
  for (int i = 0; i < Sh::NPW; ++i) {
    const int p = wave + Sh::NW * i;
    if (Sh::NW * i < Sh::NPA) voff[i] = ((unsigned)min(p >> 1, last) * (unsigned)(K / 32) + (unsigned)(p & 1)) * 1024u + (unsigned)lane * 16u;
    else voff[i] = tile_voff(p - Sh::NPA, lane, ldx, [&](int row) { return min(t0 + row, T - 1) - t0; });
  }
  f32x4 acc[RA][RB];
  if (st0 < st1) {
    if (!tile_products<P, WM, WN, RA, RB, KS, true>(acc, smem, wp + ((long)(n0 / 16) * (K / 32) + st0 * 2) * 1024,
                                                    x + (long)t0 * ldx + st0 * 64, 2048, voff, st1 - st0, wave, ks)) return;
  } else {                                                   // a slab past the last stage: its partial is zero
#pragma unroll
    for (int i = 0; i < RA; ++i)
#pragma unroll
      for (int t = 0; t < RB; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (ks) return;
  }
  const int nw = n0 + wm * RA * 16;                          // this wave's first row of W
  const unsigned strip = (unsigned)(size_t)(lds_char*)smem + (unsigned)wave * (KS == 2 ? RA * RB * 1024u : TileRows<16, RA>::BYTES);
  static_assert(TileRows<16, RA>::BYTES <= RA * RB * 1024u && TileRows<16, RA>::BYTES * Sh::NW <= Sh::LDS, "a strip per wave");
#pragma unroll
  for (int t = 0; t < RB; ++t) {
    const int tile0 = t0 + (wn * RB + t) * 16, tok = min(tile0 + j, T - 1);
    float inv = 1.f;
    if (fx.ssq_in) {
      const float* sq = fx.ssq_in + (long)tok * (fx.ssq_stride ? fx.ssq_stride : fx.ssq_groups);
      float a = 0.f;
      for (int q = 0; q < fx.ssq_groups; q += 4) { const f32x4 v = *reinterpret_cast<const f32x4*>(sq + q); a += v[0]; a += v[1]; a += v[2]; a += v[3]; }
      inv = rsqrtf(a / fx.ssq_dim + fx.eps);
    }
    if (epi == EPI_SILU) {
      unsigned d[RA];
#pragma unroll
      for (int i = 0; i < RA; ++i) {
        const f32x4 v = acc[i][t] * inv;
        const float g0 = rnd<P>(v[0]), u0 = rnd<P>(v[1]), g1 = rnd<P>(v[2]), u1 = rnd<P>(v[3]);
        d[i] = pack2<P>(rnd<P>(g0 / (1.f + __expf(-g0))) * u0, rnd<P>(g1 / (1.f + __expf(-g1))) * u1);
      }
      u16* act = reinterpret_cast<u16*>(out) + nw / 2;       // N % 16 == 0: rows of whole 16-byte groups
      tile_rows_out<4, RA>(strip, d, [&](int row, int at, u32x4 b) {
        if (tile0 + row < T && nw + at < N) *reinterpret_cast<u32x4*>(act + (long)(tile0 + row) * (N / 2) + at / 2) = b;
      });
    } else {
      f32x4 v[RA];
#pragma unroll
      for (int i = 0; i < RA; ++i) {
        v[i] = acc[i][t];
        if (epi == EPI_ROUND) { v[i] *= inv; v[i][0] = rnd<P>(v[i][0]); v[i][1] = rnd<P>(v[i][1]); v[i][2] = rnd<P>(v[i][2]); v[i][3] = rnd<P>(v[i][3]); }
      }
      tile_rows_out<16, RA>(strip, v, [&](int row, int at, u32x4 b) {
        if (tile0 + row < T && nw + at / 4 < N) *reinterpret_cast<u32x4*>(out + ((long)sp * T + tile0 + row) * N + nw + at / 4) = b;
      });
    }
  }
}

template <typename P, int WM, int WN, int RA, int RB, int KS>
__global__ __launch_bounds__(64 * WM * WN * KS, WM * WN * KS == 4 ? 2 : 1)
void dgemm_kernel(const unsigned char* __restrict__ wp, const u16* __restrict__ x, int ldx, int T, int N, int K, int S, int epi, int nbt,
                  float* __restrict__ out, GemmFused fx) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int id = tile_of_block(blockIdx.x, gridDim.x), tiles = gridDim.x / S;
  dgemm_block<P, WM, WN, RA, RB, KS>(smem, wp, x, ldx, T, N, K, S, epi, nbt, out, fx, id % tiles, id / tiles, 0);
}

// whole rounds of 256 x 256 tiles (the first `whole` workgroups), then the rows behind them in tiles of fewer tokens (tile_mix)
template <typename P, int RB>
__global__ __launch_bounds__(512, 1)
void dgemm_mixed_kernel(const unsigned char* __restrict__ wp, const u16* __restrict__ x, int ldx, int T, int N, int K, int epi, int nbt, int nbt_tail,
                        int whole, int first, float* __restrict__ out, GemmFused fx) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int b = blockIdx.x;
  if (b < whole) dgemm_block<P, 4, 2, 4, 8, 1>(smem, wp, x, ldx, T, N, K, 1, epi, nbt, out, fx, tile_of_block(b, whole), 0, 0);
  else dgemm_block<P, 4, 2, 4, RB, 1>(smem, wp, x, ldx, T, N, K, 1, epi, nbt_tail, out, fx, tile_of_block(b - whole, gridDim.x - whole), 0, first);
}

template <typename P, int RB>
static int dgemm_launch_mixed(const void* wp, const u16* x, int ldx, float* out, int T, int N, int K, int epi, int columns, const GemmFused& fx, hipStream_t st) {
  typedef TileShape<4, 2, 4, 8, 1> Sh;
  typedef TileShape<4, 2, 4, RB, 1> Tail;
  constexpr int LDS = (int)(Sh::LDS > Tail::LDS ? Sh::LDS : Tail::LDS);
  static bool attr_done[64] = {};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 64 && !attr_done[dev]) {
    if (hipFuncSetAttribute((const void*)dgemm_mixed_kernel<P, RB>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return UMB_EHIP;
    attr_done[dev] = true;
  }
  const int first = columns * Sh::BN, nbt = (T + Sh::BT - 1) / Sh::BT, nbt_tail = (T + Tail::BT - 1) / Tail::BT, whole = columns * nbt;
  hipLaunchKernelGGL((dgemm_mixed_kernel<P, RB>), dim3((unsigned)whole + (N - first + Sh::BN - 1) / Sh::BN * nbt_tail), dim3(512), LDS, st,
                     (const unsigned char*)wp, x, ldx, T, N, K, epi, nbt, nbt_tail, whole, first, out, fx);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

template <typename P, int WM, int WN, int RA, int RB, int KS>
static int dgemm_launch(const void* wp, const u16* x, int ldx, float* out, int T, int N, int K, int S, int epi, const GemmFused& fx, hipStream_t st) {
  typedef TileShape<WM, WN, RA, RB, KS> Sh;
  static bool attr_done[64] = {};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 64 && !attr_done[dev]) {
    if (hipFuncSetAttribute((const void*)dgemm_kernel<P, WM, WN, RA, RB, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Sh::LDS) != hipSuccess)
      return UMB_EHIP;
    attr_done[dev] = true;
  }
  const int nbt = (T + Sh::BT - 1) / Sh::BT;
  hipLaunchKernelGGL((dgemm_kernel<P, WM, WN, RA, RB, KS>), dim3((unsigned)((N + Sh::BN - 1) / Sh::BN) * nbt * S), dim3(64 * Sh::NW * KS), Sh::LDS, st,
                     (const unsigned char*)wp, x, ldx, T, N, K, S, epi, nbt, out, fx);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// Up to 128 tokens what a tile decides besides its time is whether K is split over two groups of waves, and so the order in which K is summed: that of
// recorded greedy continuations behind 96-token prompts, whose near-ties another rounding of the cached keys would decide otherwise.  So the tiles
// there are chosen as they were when those were recorded: five of them, by rounds x stages and the stage times of two-slot rings (only their order
// counts now, the rings are deeper).  128 is where those prompts end, not where another rule begins to pay: by tile_kind the same launches take as
// long, but for many rows in few rounds (us, this / tile_kind's, 65 / 128 tokens: gate/up 28672 x 4096 63.7 / 65.1 against 50.9 / 60.7, 32000 x 4096 65.9 / 67.5
// against 56.9 / 60.4, 6144 x 4096 in four slabs 19.4 / 20.4 against 15.8 / 17.5; 4096 x 4096, 4096 x 14336, 3072 x 2048, 2048 x 8192 within 2 %).
enum { NARROW_256 = 0, NARROW_160 = 1, NARROW_128 = 2, NARROW_128K = 3, NARROW_64K = 4, NARROW_KINDS = 5 };
static int dgemm_narrow(int T, int N, int K, int S, double* us) {
  static const struct { int bn, bt; double us; bool ksplit; } kind[NARROW_KINDS] = {
      {256, 256, 1.5, false}, {256, 160, 1.1, false}, {128, 128, 0.52, false}, {128, 128, 0.56, true}, {128, 64, 0.39, true}};
  const bool even = K % (128 * S) == 0;
  int best = NARROW_128;
  *us = 1e30;
  for (int i = 0; i < NARROW_KINDS; ++i) {
    const long wgs = (long)((N + kind[i].bn - 1) / kind[i].bn) * ((T + kind[i].bt - 1) / kind[i].bt) * S, rounds = (wgs + 255) / 256;
    if (kind[i].ksplit && (rounds > 1 || !even)) continue;
    // a lone workgroup of the two-per-CU form leaves half the wave slots empty
    const double cost = rounds * ((K / 64 + S - 1) / S) * (i == NARROW_128 && rounds == 1 ? 0.62 : kind[i].us) + 4.0;
    if (cost < *us) { *us = cost; best = i; }
  }
  return best;
}

// the tile by tile_kind (gemm_tile.h)
static int dgemm_tile(int T, int N, int K, int S, double* us = nullptr) { return tile_kind(T, N, (K / 64 + S - 1) / S, S, K % (128 * S) == 0, us, TILE_KINDS); }

extern "C" int umb_gemm_tile_kind(int T, int N, int K, int S) {
  if (T <= 128 || N < 1 || K < 64 || S < 1) return UMB_EINVAL;
  return dgemm_tile(T, N, K, S);
}

template <typename P>
static int dgemm_any(const void* wp, const u16* x, int ldx, float* out, int T, int N, int K, int S, int epi, const GemmFused& fx, hipStream_t st) {
  if (T <= 128) {
    double us;
    switch (dgemm_narrow(T, N, K, S, &us)) {
      case NARROW_256: return dgemm_launch<P, 4, 2, 4, 8, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
      case NARROW_160: return dgemm_launch<P, 4, 2, 4, 5, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
      case NARROW_128: return dgemm_launch<P, 2, 2, 4, 4, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
      case NARROW_128K: return dgemm_launch<P, 2, 2, 4, 4, 2>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
      default: return dgemm_launch<P, 2, 2, 4, 2, 2>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    }
  }
  double us;
  const int kind = dgemm_tile(T, N, K, S, &us);
  if (S == 1) {
    const TileMix mix = tile_mix(T, N, K / 64, us);
#define MIXED(KIND, RB) if (mix.columns && mix.tail == KIND) return dgemm_launch_mixed<P, RB>(wp, x, ldx, out, T, N, K, epi, mix.columns, fx, st)
    MIXED(TILE_192, 6);
    MIXED(TILE_160, 5);
    MIXED(TILE_128W, 4);
    MIXED(TILE_96, 3);
#undef MIXED
  }
  switch (kind) {
    case TILE_288: return dgemm_launch<P, 4, 2, 4, 9, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    case TILE_256: return dgemm_launch<P, 4, 2, 4, 8, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    case TILE_192: return dgemm_launch<P, 4, 2, 4, 6, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    case TILE_160: return dgemm_launch<P, 4, 2, 4, 5, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    case TILE_128W: return dgemm_launch<P, 4, 2, 4, 4, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    case TILE_96: return dgemm_launch<P, 4, 2, 4, 3, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    case TILE_128: return dgemm_launch<P, 2, 4, 4, 2, 1>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
    default: return dgemm_launch<P, 2, 2, 4, 2, 2>(wp, x, ldx, out, T, N, K, S, epi, fx, st);
  }
}

// Up to 128 tokens against more weights than the last-level cache holds the product is bound by HBM, and gemm.hip's register-resident
// kernel streams them faster (128256 x 4096, 100 tokens: 195 us, 217 here; 160 tokens: 377, 250 here).  It holds up to 144 tokens in one pass,
// and stays ahead there where the 256-row tiles of such a launch are more than one per compute unit (129 tokens, it / here: 128256 x 4096 198 /
// 245 us, 73728 x 4608 192 / 219, 128256 x 2048 111 / 122; 65536 x 5120, one round, 175 / 145; 145 tokens 377 / 245).  Less weight of such a
// launch already stays ahead there (65 tokens, 100352 x 2560 101 / 125) unless K is short (256000 x 1024 127 / 117).
bool umb_dgemm_ok(const void* x, const void* out, int ldx, int T, int N, int K, int S, int epi) {
  static const bool off = getenv("UMB_NO_VGEMM") != nullptr || getenv("UMB_VGEMM_PLAIN") != nullptr;     // gemm.hip's diagnostics
  const long bytes = (long)N * K * 2;
  const bool streams = (T <= 128 && bytes > (512L << 20)) || (T <= 144 && N > 65536 && K >= 1536 && bytes > (448L << 20));
  return !off && T > 64 && K % 64 == 0 && N % 16 == 0 && ldx % 8 == 0 && ((uintptr_t)x | (uintptr_t)out) % 16 == 0 && epi <= EPI_SILU &&
         (long)ldx * 512 < (1L << 31) && !streams;
}

// K slabs of a wide dense product whose partials are summed by the kernel behind it: the least of the product's time and of what reading the
// partials beyond the first costs there (8 TB/s: they come from the last-level cache).  1024 tokens: 6144 x 4096 S = 1, 4096 x 14336 S = 4 in 256 x 256
// tiles (93 us and 13.1 in the residual behind it; S = 2 in 256 x 128 102 and 10.3; whole 190)
int umb_dgemm_split(int T, int N, int K, int S_plan) {
  int best_s = 1;
  double best = 1e30, us = 0.0;
  for (int S = 1; S <= S_plan && S <= K / 128 && (long)S * T * N * 4 < (1L << 31); ++S) {
    if (T <= 128) (void)dgemm_narrow(T, N, K, S, &us);
    else (void)dgemm_tile(T, N, K, S, &us);
    const double cost = us + (S - 1) * (double)T * N * 4 / (T <= 128 ? 3e6 : 8e6);
    if (cost < best) { best = cost; best_s = S; }
  }
  return best_s;
}

int umb_dgemm(const void* wp, const u16* x, int ldx, float* out, int T, int N, int K, int S, int epi, const GemmFused& fx, int dtype,
              hipStream_t st) {
  DISPATCH_DTYPE(dtype, { return dgemm_any<P>(wp, x, ldx, out, T, N, K, S, epi, fx, st); })
}
