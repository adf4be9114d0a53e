// Main loop of the LDS-staged 16-bit matrix products whose operands are both re-used many times (prompts, wide verification):
// acc = A[rows][K] . B[tokens][K]^T, a workgroup's tile of WM RA x WN RB 16 x 16 products, fp32 accumulation in k order.
//
// What bounds it is the path from LDS to the matrix pipes: a wave of RA x RB products reads RA + RB fragments (1 KiB each) per 32 k
// for RA RB products of 16 cycles, and a CU's LDS delivers one KiB in 8 cycles.  64 x 64 outputs per wave (4 x 4) ask for all of
// it, 64 x 128 (4 x 8) for three quarters.  Hence:
//   * operands go HBM / L2 -> LDS by LDS-DMA (1-KiB pieces of 8 rows x 128 B: whole lines, no VGPR on the way, no address arithmetic
//     in the loop); the 16-byte column of a row is XOR-swizzled on the SOURCE side, so fragment reads meet no bank conflict;
//   * a ring of two to four slots of 64 k for each operand, as many as the LDS holds.  ONE barrier per stage stands between its two 32-k
//     phases: when a wave arrives there it has every fragment of the stage in registers, so behind the barrier the slot is free for the
//     stage a ring's length further on, and the next stage (whose pieces every wave has waited for) can be read: the fragments of a phase are
//     requested, one per few products, while the products of the phase before run, across the stage boundary too.  With two slots the
//     pieces that are asked for last have half a stage to arrive, and no stage is shorter than the 1.0 us that they take from L2: 256 x 128 outputs
//     1.05 -> 0.86 us a stage with three, 256 x 160 1.1 -> 0.95 - 1.05, 128 x 128 (eight waves, four slots; before: K over two groups of four,
//     0.55) 0.49.  256 x 256 and 256 x 192 outputs have no room for three of both, but for three of A (the weights, which come from further away) and two
//     of B, whose pieces are then asked for first: 1.47 -> 1.36 and 1.36 -> 1.19 us a stage (K 4096 -> 8192, 256 workgroups; on zeros, without the
//     power limit, 2048 x 8192 x 4096 91 -> 78 us; 1024 x 28672 x 4096 197 -> 192).  Four waves of 128 x 128 outputs (a third less LDS traffic, sums in
//     AGPRs) on the same rings: 105 us where these take 101, 88 on zeros.
//   * the last stages ask for nothing: pieces past the end would be waited for behind the last product.
// K-split (KS = 2): two groups of WM x WN waves take alternate stages in slots of their own and their tiles are added (group 0 +
// group 1) at the end: two waves per SIMD where a launch has at most one workgroup per CU.
// Measured against the register-staged kernel it replaces (bf16, random data, one MI355X; both sides in seq_linear.hip).
#pragma once
#include "common.h"
#include <type_traits>

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) float lds_f32;

// one LDS-DMA piece: 64 lanes x 16 B, global address = sbase + voff (per lane), LDS address = ldsaddr + 16 * lane
__device__ __forceinline__ void tile_dma(unsigned voff, const void* sbase, unsigned ldsaddr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(sbase), "s"(ldsaddr) : "memory", "m0");
}

// the same for what is read once: not kept in L2 in the place of what is
__device__ __forceinline__ void tile_dma_once(unsigned voff, const void* sbase, unsigned ldsaddr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
               :: "v"(voff), "s"(sbase), "s"(ldsaddr) : "memory", "m0");
}

// a KiB's lines on their way to L2: a word of every 16 bytes to LDS that nobody reads
__device__ __forceinline__ void tile_touch(unsigned voff, const void* sbase, unsigned ldsaddr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               :: "v"(voff), "s"(sbase), "s"(ldsaddr) : "memory", "m0");
}

template <int WM, int WN, int RA, int RB, int KS> struct TileShape {
  static constexpr int NW = WM * WN;                          // waves of one K group
  static constexpr int BN = 16 * WM * RA, BT = 16 * WN * RB;  // rows of A, tokens of B
  static constexpr int NPA = BN / 8, NPB = BT / 8;            // 1-KiB pieces of a stage
  static constexpr int NPW = (NPA + NPB + NW - 1) / NW;       // pieces a wave fetches per stage
  static constexpr unsigned SA = NPA * 1024u, SB = NPB * 1024u, SLOT = SA + SB;
  static constexpr int PER_CU = NW * KS == 4 ? 2 : 1;         // workgroups that share a CU
  // where the pieces do not deal out evenly, a wave without a last piece of its own fetches into the KiB behind the slots
  static constexpr bool EVEN = (NPA + NPB) % NW == 0;
  static constexpr unsigned ROOM = 160u * 1024 / PER_CU - (EVEN ? 0 : 1024);
  static constexpr int FIT = (int)(ROOM / (KS * SLOT)), NSB = FIT < 4 ? FIT : 4;               // slots of B's ring
  static constexpr int NSA = NSB == 2 && KS * (3 * SA + 2 * SB) <= ROOM ? 3 : NSB;             // and of A's
  static constexpr unsigned RINGS = NSA * SA + NSB * SB;
  static constexpr size_t LDS = (size_t)KS * RINGS + (EVEN ? 0 : 1024);
  static_assert(NSB >= 2 && NPA % NW == 0 && (EVEN || KS == 1) && (KS == 1 || RA * RB * NW * 1024u <= LDS), "whole rounds of A pieces; a group's tile fits the slots");
};

// The tiles a launch chooses from, and what a 64-k stage of a whole round of 256 workgroups takes (us; one MI355X, bf16, random data).  Few sizes
// of a prompt fill rounds of one tile; between 0.46 (256 x 256) and 1.4 ns a stage, row and token the right one is the one that fills best.
// (Of one whole round, between K 4096 and 8192, the first two are down to 1.36 and 1.19 with three slots of A; the rules were fitted with these.)
//                       rows tokens stage
enum { TILE_256 = 0,  //  256   256  1.42
       TILE_192 = 1,  //  256   192  1.20
       TILE_160 = 2,  //  256   160  1.04
       TILE_128W = 3, //  256   128  0.86
       TILE_96 = 4,   //  256    96  0.73
       TILE_128 = 5,  //  128   128  0.49
       TILE_64K = 6,  //  128    64  0.38   K over two groups of waves
       TILE_288 = 7,  //  256   288  2.06   A in fragments: tokens that fill 288s in fewer rounds, us before / with it: 257 of 128256 x 8192 650 / 565 (two tiles of
                      //                    160), 288 of x 4096 330 / 299, gate/up 28672 x 4096 of 513 138 / 117, 16384 x 2048 of 1130 78 / 68, 8192 x 4096 of 2250 142 / 120
       TILE_KINDS = 8 };
struct Tile { int bn, bt; double us; };
constexpr Tile TILES[TILE_KINDS] = {{256, 256, 1.42}, {256, 192, 1.20}, {256, 160, 1.04}, {256, 128, 0.86}, {256, 96, 0.73}, {128, 128, 0.49}, {128, 64, 0.38}, {256, 288, 2.06}};
// us of a launch: 4, and for each round its stages, 2 in front of them and 14 for 256 x 256 outputs behind them; a last round that is not
// full takes a little less (its share of the memory path is larger).  rows: of A; stages: of one slab; S: slabs
static inline double tile_cost(int kind, int T, int rows, int stages, int S) {
  const Tile k = TILES[kind];
  const long wgs = (long)((rows + k.bn - 1) / k.bn) * ((T + k.bt - 1) / k.bt) * S, rest = wgs % 256;
  const double load = rest / 256.0, products = stages * k.us, out = 2.1e-4 * k.bn * k.bt;
  return 4.0 + (wgs / 256) * (products + out + 2.0) + (rest ? products * (0.8 + 0.2 * load) + out * load + 2.0 : 0.0);
}
// The least of them (the K-split one takes an even number of stages); kinds: TILE_288 too where A lies in fragments, with K whole or in slabs of five stages and
// more: in shorter ones its two slots of B stand bare (those that the costs give to it, time without / with it: K whole 1.12 in the mean, 2094 of 2106 0.97 or more; slabs
// of five stages and more 1.10, 2001 of 2066; shorter ones 1.03, a sixth of them under 0.97, 280 tokens of 22432 x 512 in three slabs 29.2 / 37.7 us).
static inline int tile_kind(int T, int rows, int stages, int S, bool even, double* us = nullptr, int kinds = TILE_288) {
  int best = 0;
  for (int i = 1; i < kinds; ++i)
    if ((i != TILE_64K || even) && (i != TILE_288 || S == 1 || stages >= 5) && tile_cost(i, T, rows, stages, S) < tile_cost(best, T, rows, stages, S)) best = i;
  if (us) *us = tile_cost(best, T, rows, stages, S);
  return best;
}

// More 256 x 256 tiles than whole rounds of 256 workgroups: the whole rounds take the first `columns` 256-row columns, the columns that are left go in
// tiles of `tail`'s tokens (256 rows too) behind them in the same launch, chosen as above (the first of them run beside the last round's end).  columns 0: no.
// What it may save is the last round's idle share, so it has to be 3 % ahead.
struct TileMix { int columns, tail; };
static inline TileMix tile_mix(int T, int rows, int stages, double single) {
  const long nbt = (T + 255) / 256, all = (rows + 255L) / 256 * nbt, rounds = all / 256;
  TileMix best{0, 0};
  if (rounds == 0 || all % 256 == 0 || nbt > 256) return best;
  const int columns = (int)(256 * rounds / nbt);
  const long tail = (rows + 255) / 256 - columns, spare = 256 * rounds - columns * nbt;
  if (tail <= 0) return best;
  const double main = 4.0 + rounds * (stages * TILES[TILE_256].us + 2.1e-4 * 256 * 256 + 2.0);
  double least = 0.97 * single;
  for (int i = TILE_192; i <= TILE_96; ++i) {              // the others of 256 rows
    const Tile k = TILES[i];
    const long wgs = tail * ((T + k.bt - 1) / k.bt) - spare, rest = wgs > 0 ? wgs % 256 : 0;
    const double load = rest / 256.0, products = stages * k.us, out = 2.1e-4 * 256 * k.bt;
    const double us = main + (wgs > 0 ? wgs / 256 * (products + out + 2.0) : 0.0) + (rest ? products * (0.8 + 0.2 * load) + out * load + 2.0 : 0.0);
    if (us < least) { least = us; best = TileMix{columns, i}; }
  }
  return best;
}

// Row block of a workgroup: the hardware deals consecutive workgroups to the eight XCDs in turn; here the workgroups of one XCD get
// consecutive tile numbers, so that the tiles its L2 serves share operand rows.
__device__ __forceinline__ int tile_of_block(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, xcd = b & 7;
  return xcd * q + min(xcd, r) + (b >> 3);
}

// piece p (8 rows) of an operand stored [rows][K]: lane l fetches row 8 p + l / 8, 16-byte column (l % 8) ^ (l / 8); row_of maps the
// tile's row to a row of the operand counted from its base
template <typename F> __device__ __forceinline__ unsigned tile_voff(int p, int lane, int ld, F row_of) {
  const int r = lane >> 3, c = (lane & 7) ^ r;
  return ((unsigned)row_of(p * 8 + r) * (unsigned)ld + c * 8u) * 2u;
}

// abase / bbase: the operands at k = 0 of the tile (a stage advances them by astep / 128 bytes); voff: per-lane byte offsets of this
// wave's pieces (NPA / NW of A, then those of B).  FRAG: A lies in 1-KiB fragments already (lane l's 16 bytes at 16 l): its pieces are
// the fragments (16 rows, 32 k) in the order row tile, k half.  nst: stages of 64 k (a multiple of KS).  On return acc is complete in
// the waves of group 0, which may use their share of LDS from then on (16 RA RB KiB / 16 a wave with a K split, else LDS / NW); returns whether
// this wave is one of them.
template <typename P, int WM, int WN, int RA, int RB, int KS, bool FRAG>
__device__ __forceinline__ bool tile_products(f32x4 (&acc)[RA][RB], unsigned char* smem, const void* abase, const void* bbase, long astep,
                                              const unsigned (&voff)[TileShape<WM, WN, RA, RB, KS>::NPW], int nst, int wave, int ks) {
  typedef TileShape<WM, WN, RA, RB, KS> S;
  constexpr int NW = S::NW, NPA = S::NPA, NPW = S::NPW, PA = NPA / NW, PB = NPW - PA, NF = RA + RB, NM = RA * RB, NSA = S::NSA, NSB = S::NSB;
  // 144 sums a lane: the fragments of two phases are too many beside them, so B's are given up one by one (A's innermost) while the next are read, one
  // per 2.8 products, and A's offsets stand in scalar registers (59 values spilled without, now 3)
  constexpr bool SPREAD = RB > 8;
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
  const unsigned lds0 = (unsigned)(size_t)(lds_char*)smem + (unsigned)ks * S::RINGS, lds1 = lds0 + NSA * S::SA;
  const int n = nst / KS;                                     // stages of this group
  unsigned aoff[PA];                                          // fragments: a piece's offset is the wave's, its lanes 16 bytes apart
#pragma unroll
  for (int i = 0; i < PA; ++i) aoff[i] = SPREAD && FRAG ? __builtin_amdgcn_readfirstlane(voff[i]) : 0;
  auto issue = [&](int st, unsigned slot, int i) {            // pieces 0 .. PA - 1 are A's; slot: of the ring they go to
    const unsigned p = (unsigned)(wave + NW * i);
    unsigned dst = i < PA ? lds0 + slot + p * 1024u : lds1 + slot + (p - NPA) * 1024u;
    if (!S::EVEN && i == NPW - 1 && wave + NW * i >= NPA + S::NPB) dst = lds0 + S::RINGS;
    const long s = (long)min(st, n - 1) * KS + ks;
    if (SPREAD && FRAG && i < PA) tile_dma((unsigned)lane * 16u, static_cast<const char*>(abase) + s * astep + aoff[i], dst);
    else if (i < PA) tile_dma(voff[i], static_cast<const char*>(abase) + s * astep, dst);
    else tile_dma(voff[i], static_cast<const char*>(bbase) + s * 128, dst);
  };
  // Two slots leave a piece of A less than a stage, and it may come from memory: its lines are asked for a stage and a half earlier (with a
  // head of 257 tokens 72 - 89 us off a whole call, 55 without)
  constexpr bool TOUCH = SPREAD && FRAG;
  static_assert(!TOUCH || !S::EVEN, "a KiB of nobody's");
  auto touch = [&](int st, int i) {
    tile_touch((unsigned)lane * 16u, static_cast<const char*>(abase) + ((long)min(st, n - 1) * KS + ks) * astep + aoff[i], lds0 + S::RINGS);
  };
  // fragment (16 rows, 32 k) of two row pieces: lane (j, g) reads row j, 16-byte column 4 kh + g
  unsigned foff[2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) foff[kh] = (unsigned)((j >> 3) * 1024 + ((j & 7) * 8 + ((kh * 4 + g) ^ (j & 7))) * 16);
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int t = 0; t < RB; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 fa[2][RA], fb[2][RB];
  auto read = [&](unsigned sa, unsigned sb, int kh, int i) {  // the i-th fragment of a phase, in the order the products want them
    const unsigned ao = lds0 + sa + (FRAG ? (unsigned)(kh * 1024 + lane * 16) : foff[kh]), bo = lds1 + sb + foff[kh];
    if (SPREAD) {
      if (i < RA) fa[kh][i] = *reinterpret_cast<const lds_u32x4*>((size_t)(ao + (unsigned)(wm * RA + i) * 2048u));
      else fb[kh][i - RA] = *reinterpret_cast<const lds_u32x4*>((size_t)(bo + (unsigned)(wn * RB + i - RA) * 2048u));
    } else if (i == 0) fa[kh][0] = *reinterpret_cast<const lds_u32x4*>((size_t)(ao + (unsigned)(wm * RA) * 2048u));
    else if (i <= RB) fb[kh][i - 1] = *reinterpret_cast<const lds_u32x4*>((size_t)(bo + (unsigned)(wn * RB + i - 1) * 2048u));
    else fa[kh][i - RB] = *reinterpret_cast<const lds_u32x4*>((size_t)(ao + (unsigned)(wm * RA + i - RB) * 2048u));
  };
  unsigned sa = 0, sb = 0, na = S::SA, nb = S::SB;            // slots of the stage whose products run, and of the one behind it
  // the products of one half of stage st; FETCH: 2 the stages NSA and NSB further on are asked for (behind the barrier), 1 B's alone, 0 none
  auto phase = [&](auto half, auto fetch, auto more, int st) {
    constexpr int KH = decltype(half)::value, FETCH = decltype(fetch)::value;
    constexpr bool READ = KH == 0 || decltype(more)::value;
    constexpr int GAP = NM / NF > 0 ? NM / NF : 1, DG = NM / NPW > 0 ? NM / NPW : 1;   // products per fragment read, per piece
    static_assert(GAP * (NF - 1) < NM && DG * (NPW - 1) < NM, "every read and every piece has a product to hide behind");
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if constexpr (SPREAD) {
        if (READ && (m == 0 || m * NF / NM != (m - 1) * NF / NM)) read(KH == 0 ? sa : na, KH == 0 ? sb : nb, KH ^ 1, m * NF / NM);
      } else if (READ && m % GAP == 0 && m / GAP < NF) read(KH == 0 ? sa : na, KH == 0 ? sb : nb, KH ^ 1, m / GAP);
      if (TOUCH && KH == 0 && FETCH > 1 && m % (NM / PA) == 1 && m / (NM / PA) < PA) touch(st + NSA + 1, m / (NM / PA));
      if (KH == 1 && m % DG == 0 && m / DG < NPW) {
        const int i = NSA > NSB ? (m / DG < PB ? PA + m / DG : m / DG - PB) : m / DG;            // the shorter ring's pieces first
        if (i >= PA ? FETCH > 0 : FETCH > 1) issue(st + (i < PA ? NSA : NSB), i < PA ? sa : sb, i);
      }
      const int r = SPREAD ? m % RA : m / RB, t = SPREAD ? m / RA : m % RB;
      acc[r][t] = P::mfma(fa[KH][r], fb[KH][t], acc[r][t]);
      if (SPREAD || (m + 1) % GAP == 0) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // a stage; LEFT: what may still be on its way when its successor has to be there
  auto stage = [&](auto left, auto fetch, auto more, int st) {
    phase(std::integral_constant<int, 0>{}, fetch, more, st);
    // every fragment of stage st is in registers, and this wave's pieces of stage st + 1 are in LDS
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(decltype(left)::value) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    phase(std::integral_constant<int, 1>{}, fetch, more, st);
    sa = na;
    sb = nb;
    na = na == (NSA - 1) * S::SA ? 0u : na + S::SA;
    nb = nb == (NSB - 1) * S::SB ? 0u : nb + S::SB;
  };
#pragma unroll
  for (int c = 0; c < NSA; ++c)
#pragma unroll
    for (int i = 0; i < NPW; ++i)
      if (i < PA || c < NSB) issue(c, c * (i < PA ? S::SA : S::SB), i);
  constexpr int ALONE = NSA > NSB ? PA : 0;                   // A's pieces of the stage that only its ring holds
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NSB - 1) * NPW + ALONE) : "memory");
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < NF; ++i) read(0, 0, 0, i);
  int st = 0;
  for (; st < n - NSA; ++st) stage(std::integral_constant<int, (NSB - 2) * NPW + ALONE + (TOUCH ? PA : 0)>{}, std::integral_constant<int, 2>{}, std::true_type{}, st);
  // the last NSA stages: nothing is asked for that no stage will use
  auto last = [&](auto t_) {
    constexpr int t = decltype(t_)::value, LEFT = (NSB - 2 - t > 0 ? NSB - 2 - t : 0) * NPW + (t == 0 ? ALONE : 0);
    if (st < n) stage(std::integral_constant<int, LEFT>{}, std::integral_constant<int, (t < NSA - NSB)>{}, std::integral_constant<bool, (t < NSA - 1)>{}, st);
    ++st;
  };
  last(std::integral_constant<int, 0>{});
  last(std::integral_constant<int, 1>{});
  if constexpr (NSA > 2) last(std::integral_constant<int, 2>{});
  if constexpr (NSA > 3) last(std::integral_constant<int, 3>{});
  static_assert(NSA >= 2 && NSA <= 4 && (NSA == NSB || (NSA == 3 && NSB == 2)), "the last stages above");
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // nothing of this wave may still be writing LDS
  __builtin_amdgcn_s_barrier();                                 // and none reads a slot any more
  if constexpr (KS == 2) {
    f32x4* red = reinterpret_cast<f32x4*>(smem) + wave * NM * 64 + lane;
    if (ks == 1) {
#pragma unroll
      for (int i = 0; i < NM; ++i) red[i * 64] = acc[i / RB][i % RB];
    }
    __syncthreads();
    if (ks == 1) return false;
#pragma unroll
    for (int i = 0; i < NM; ++i) acc[i / RB][i % RB] += red[i * 64];
  }
  return true;
}

// Outputs of one token tile of a wave, on their way to rows of memory.  After the products lane (j, g) holds, for each of NI row tiles, the QB
// bytes of token j behind 4 g outputs: stored from there, an instruction writes 16 rows of 4 QB bytes with neighbouring lanes on different
// rows, and the stores of a launch take as long as a third of its products (8192 x 2048 outputs, K = 2048, bf16: 72 us, 48 without
// stores).  Through a strip of LDS of the wave's own they leave as whole lines: put(row, byte, 16 bytes) with neighbouring lanes on
// neighbouring bytes.  `strip`: its LDS address, TileRows::BYTES of it; rows of it are 16 bytes more than the data apart.
template <int QB, int NI> struct TileRows {
  static constexpr int ROW = NI * 4 * QB, STRIDE = ROW + 16, LPR = ROW / 16, RPI = 64 / LPR;       // lanes a row, rows an instruction
  static constexpr unsigned BYTES = 16u * STRIDE;
  static_assert(ROW % 16 == 0 && 64 % LPR == 0 && 16 % RPI == 0, "whole rows");
};
template <int QB, int NI, typename V, typename Put>
__device__ __forceinline__ void tile_rows_out(unsigned strip, const V (&v)[NI], Put put) {
  typedef TileRows<QB, NI> R;
  typedef __attribute__((address_space(3))) V lds_v;
  static_assert(sizeof(V) == QB, "a lane's bytes of a row tile");
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
#pragma unroll
  for (int i = 0; i < NI; ++i) *reinterpret_cast<lds_v*>((size_t)(strip + (unsigned)(j * R::STRIDE + (i * 4 + g) * QB))) = v[i];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int k = 0; k < 16 / R::RPI; ++k) {
    const int row = k * R::RPI + lane / R::LPR, at = lane % R::LPR * 16;
    put(row, at, *reinterpret_cast<const lds_u32x4*>((size_t)(strip + (unsigned)(row * R::STRIDE + at))));
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
