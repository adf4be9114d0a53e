// Main loop of the LDS-staged 16-bit matrix products whose operands are both re-used many times (prompts, wide verification):
// acc = A[rows][K] . B[tokens][K]^T, a workgroup's tile of WM RA x WN RB 16 x 16 products, fp32 accumulation in k order.
//
// What bounds it is the path from LDS to the matrix pipes: a wave of RA x RB products reads RA + RB fragments (1 KiB each) per 32 k
// for RA RB products of 16 cycles, and a CU's LDS delivers one KiB in 8 cycles.  64 x 64 outputs per wave (4 x 4) ask for all of
// it, 64 x 128 (4 x 8) for three quarters.  Hence:
//   * operands go HBM / L2 -> LDS by LDS-DMA (1-KiB pieces of 8 rows x 128 B: whole lines, no VGPR on the way, no address arithmetic
//     in the loop); the 16-byte column of a row is XOR-swizzled on the SOURCE side, so fragment reads meet no bank conflict;
//   * two slots of 64 k.  ONE barrier per stage stands between its two 32-k phases: when a wave arrives there it has every fragment
//     of the stage in registers, so behind the barrier the slot is free for the stage after the next, and the next stage (whose
//     pieces every wave has waited for) can be read: the fragments of a phase are requested, one per few products, while the
//     products of the phase before run, across the stage boundary too, and a stage's pieces have a whole stage to arrive.
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

template <int WM, int WN, int RA, int RB, int KS> struct TileShape {
  static constexpr int NW = WM * WN;                          // waves of one K group
  static constexpr int BN = 16 * WM * RA, BT = 16 * WN * RB;  // rows of A, tokens of B
  static constexpr int NPA = BN / 8, NPB = BT / 8;            // 1-KiB pieces of a stage
  static constexpr int NPW = (NPA + NPB + NW - 1) / NW;       // pieces a wave fetches per stage
  static constexpr unsigned SLOT = (NPA + NPB) * 1024u;
  // where the pieces do not deal out evenly, a wave without a last piece of its own fetches into the KiB behind the slots
  static constexpr bool EVEN = (NPA + NPB) % NW == 0;
  static constexpr size_t LDS = (size_t)KS * 2 * SLOT + (EVEN ? 0 : 1024);
  static_assert(NPA % NW == 0 && (EVEN || KS == 1) && (KS == 1 || RA * RB * NW * 1024u <= LDS), "whole rounds of A pieces; a group's tile fits the slots");
};

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
// the waves of group 0; returns whether this wave is one of them.
template <typename P, int WM, int WN, int RA, int RB, int KS, bool FRAG>
__device__ __forceinline__ bool tile_products(f32x4 (&acc)[RA][RB], unsigned char* smem, const void* abase, const void* bbase, long astep,
                                              const unsigned (&voff)[TileShape<WM, WN, RA, RB, KS>::NPW], int nst, int wave, int ks) {
  typedef TileShape<WM, WN, RA, RB, KS> S;
  constexpr int NW = S::NW, NPA = S::NPA, NPW = S::NPW, NF = RA + RB, NM = RA * RB;
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
  const unsigned lds0 = (unsigned)(size_t)(lds_char*)smem + (unsigned)ks * 2u * S::SLOT;
  const int n = nst / KS;                                     // stages of this group
  auto issue = [&](int st, int i) {
    unsigned dst = lds0 + (unsigned)(st & 1) * S::SLOT + (unsigned)(wave + NW * i) * 1024u;
    if (!S::EVEN && i == NPW - 1 && wave + NW * i >= NPA + S::NPB) dst = lds0 + 2u * S::SLOT;
    const long s = (long)min(st, n - 1) * KS + ks;
    if (NW * i < NPA) tile_dma(voff[i], static_cast<const char*>(abase) + s * astep, dst);
    else tile_dma(voff[i], static_cast<const char*>(bbase) + s * 128, dst);
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
  auto read = [&](int st, int kh, int i) {                    // the i-th fragment of a phase, in the order the products want them
    const unsigned base = lds0 + (unsigned)(st & 1) * S::SLOT;
    const unsigned ao = base + (FRAG ? (unsigned)(kh * 1024 + lane * 16) : foff[kh]);
    if (i == 0) fa[kh][0] = *reinterpret_cast<const lds_u32x4*>((size_t)(ao + (unsigned)(wm * RA) * 2048u));
    else if (i <= RB) fb[kh][i - 1] = *reinterpret_cast<const lds_u32x4*>((size_t)(base + foff[kh] + NPA * 1024u + (unsigned)(wn * RB + i - 1) * 2048u));
    else fa[kh][i - RB] = *reinterpret_cast<const lds_u32x4*>((size_t)(ao + (unsigned)(wm * RA + i - RB) * 2048u));
  };
  auto phase = [&](auto half, int st) {
    constexpr int KH = decltype(half)::value;
    constexpr int GAP = NM / NF > 0 ? NM / NF : 1, DG = NM / NPW > 0 ? NM / NPW : 1;   // products per fragment read, per piece
    static_assert(GAP * (NF - 1) < NM && DG * (NPW - 1) < NM, "every read and every piece has a product to hide behind");
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m % GAP == 0 && m / GAP < NF) read(KH == 0 ? st : st + 1, KH ^ 1, m / GAP);
      if (KH == 1 && m % DG == 0 && m / DG < NPW) issue(st + 2, m / DG);
      acc[m / RB][m % RB] = P::mfma(fa[KH][m / RB], fb[KH][m % RB], acc[m / RB][m % RB]);
      if ((m + 1) % GAP == 0) __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int i = 0; i < NPW; ++i) issue(0, i);
#pragma unroll
  for (int i = 0; i < NPW; ++i) issue(1, i);
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NPW) : "memory");
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < NF; ++i) read(0, 0, i);
  for (int st = 0; st < n; ++st) {
    phase(std::integral_constant<int, 0>{}, st);
    // every fragment of stage st is in registers, and this wave's pieces of stage st + 1 are in LDS
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    phase(std::integral_constant<int, 1>{}, st);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // nothing of this wave may still be writing LDS
  if constexpr (KS == 2) {
    __builtin_amdgcn_s_barrier();
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
