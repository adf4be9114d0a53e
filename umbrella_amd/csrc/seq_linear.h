// What the few-token products share (seq_linear.hip, and seq_front.hip where a norm stands in front of them): fragments, epilogues, the pieces of
// the streaming kernels and where those pay.
#pragma once
#include "gemm_tile.h"
#include "seq_common.h"

template <typename P> struct Frag8 { u32x4 v; };
template <> struct Frag8<F32> { f32x4 lo, hi; };

template <typename P, bool VEC>
__device__ __forceinline__ Frag8<P> load8(const typename El<P>::type* __restrict__ row, int k, int K) {
  Frag8<P> f;
  if constexpr (VEC) {                      // K % 8 == 0: k < K means the whole 8-group is inside, 16-byte aligned
    const bool in = k < K;
    if constexpr (sizeof(typename El<P>::type) == 2) {
      f.v = in ? *reinterpret_cast<const u32x4*>(row + k) : u32x4{0u, 0u, 0u, 0u};
    } else {
      f.lo = in ? *reinterpret_cast<const f32x4*>(row + k) : f32x4{0.f, 0.f, 0.f, 0.f};
      f.hi = in ? *reinterpret_cast<const f32x4*>(row + k + 4) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  } else {
    if constexpr (sizeof(typename El<P>::type) == 2) {
      unsigned e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = (k + i < K) ? (unsigned)row[k + i] : 0u;
      f.v = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
    } else {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = (k + i < K) ? row[k + i] : 0.f;
      f.lo = f32x4{e[0], e[1], e[2], e[3]};
      f.hi = f32x4{e[4], e[5], e[6], e[7]};
    }
  }
  return f;
}

template <typename P> __device__ __forceinline__ f32x4 mma8(const Frag8<P>& a, const Frag8<P>& b, f32x4 c) {
  return P::mfma(a.v, b.v, c);
}
template <> __device__ __forceinline__ f32x4 mma8<F32>(const Frag8<F32>& a, const Frag8<F32>& b, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.lo[i], b.lo[i], c, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.hi[i], b.hi[i], c, 0, 0, 0);
  return c;
}

enum { EPI_F32 = 0, EPI_DT = 1, EPI_SILU_MUL = 2, EPI_GATE = 3, EPI_RELU2 = 4, EPI_CLAMP_GLU = 5, EPI_GELU_MUL = 6, EPI_GATE_ROW = 7, EPI_CAP = 8 };
// the stacked-halves epilogues: silu(gate) * up, gelu(gate) * up (tanh form), or the capped form g sigmoid(alpha g) (u + 1) with
// g = min(gate, limit), u = clamp(up, -limit, limit)
static inline bool epi_dual(int epi) { return epi == EPI_SILU_MUL || epi == EPI_CLAMP_GLU || epi == EPI_GELU_MUL; }
// epilogues that umb_seq_linear / umb_seq_linear_grouped take by number (the others have constants or a gate of their own)
static inline bool epi_plain(int epi) {
  return epi == EPI_F32 || epi == EPI_DT || epi == EPI_SILU_MUL || epi == EPI_RELU2 || epi == EPI_GELU_MUL;
}
// 0.5 z (1 + tanh(u)) with u = sqrt(2 / pi) (z + 0.044715 z^3), as z / (1 + e^(-2 u)): the same function, one exponential, and no
// cancellation where tanh is near -1
__device__ __forceinline__ float gelu_tanhf_(float z) { return over_one_plus_exp(z, 1.5957691216057308f * (z + 0.044715f * z * z * z)); }
template <int EPI> __device__ __forceinline__ float glu_of(float g, float u, float limit, float alpha) {
  if constexpr (EPI == EPI_CLAMP_GLU) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return over_one_plus_exp(g, alpha * g) * (u + 1.f);
  } else if constexpr (EPI == EPI_GELU_MUL) {
    return gelu_tanhf_(g) * u;
  } else {
    return over_one_plus_exp(g, g) * u;
  }
}
__device__ __forceinline__ float glu_pair(int epi, float g, float u, float limit, float alpha) {
  if (epi == EPI_CLAMP_GLU) return glu_of<EPI_CLAMP_GLU>(g, u, limit, alpha);
  if (epi == EPI_GELU_MUL) return glu_of<EPI_GELU_MUL>(g, u, limit, alpha);
  return glu_of<EPI_SILU_MUL>(g, u, limit, alpha);
}

// Where a launch departs from the dense [T][K] x [N][K] problem: row strides of x and out, a batch of independent problems
// along blockIdx.z (element strides sx / sw / so), or token tiles read from device memory (grouped: tile blockIdx.y is
// {group, first row, rows}; its weights start at w + group * gs).  EPI_GATE multiplies by sigmoid(gate[t ldg + z sg + n]),
// EPI_GATE_ROW by sigmoid(gate[t ldg + z sg]): one number per row and problem.
struct LinExt {
  int ldx, ldo;
  // streaming kernel.  parts > 1: blockIdx.z is a slab of K and not a problem, part_chunks 512-byte chunks (one more in the first ones); its sums go to
  // out + z so, the bias into slab 0's.  step: distance of a workgroup's row blocks (gridDim.x, read with the other arguments); turn: first_chunk
  int parts, part_chunks, step, turn;
  long sx, sw, so, gs;
  const int* tiles;
  const float* gate;
  int ldg, sg;
  float limit, alpha;      // EPI_CLAMP_GLU; EPI_CAP: out = limit tanh(acc / limit), fp32
};
static inline LinExt lin_dense(int N, int K) { return LinExt{K, N, 0, 0, 0, 0, 0, 0, 0, 0, nullptr, nullptr, 0, 0, 0.f, 0.f}; }

template <int NT, int TT, int BP, bool DUAL, int R> struct StreamShape {     // BP: token pieces (8 TT, fewer for very few tokens)
  static constexpr int AP = (DUAL ? 16 : 8) * NT, NP = AP + BP, PW = (NP + 3) / 4, AT = DUAL ? 2 * NT : NT;
  static constexpr unsigned PIECE = 1040u, SLOT = NP * PIECE;
  static constexpr size_t RED = (size_t)AT * 4 * TT * 1024, LDS = (size_t)R * SLOT + (NP % 4 ? PIECE : 0);
  static_assert(AP % 4 == 0 && R >= 2 && LDS <= 160 * 1024 && RED <= SLOT, "whole rounds of weight pieces; the CU's LDS");
  static_assert(BP % TT == 0 && (BP == 8 * TT || TT == 1), "token tiles of whole pieces");
  // place of a tile's row inside a slot; a token tile staged in part repeats its pieces: columns that are not stored
  static constexpr unsigned row_at(int first_piece, int pieces, int row) { return (unsigned)(first_piece + (row >> 1) % pieces) * PIECE + (unsigned)(row & 1) * 512u; }
  static constexpr unsigned weight_row(int tile, int row) { return row_at(8 * tile, 8, row); }
  static constexpr unsigned token_row(int tile, int row) { return row_at(AP + 8 * tile, BP / TT, row); }
  static constexpr bool rows_inside_slot() {
    for (int row = 0; row < 16; ++row) {
      for (int i = 0; i < AT; ++i) if (weight_row(i, row) + 512u > (unsigned)AP * PIECE) return false;
      for (int i = 0; i < TT; ++i) if (token_row(i, row) < (unsigned)AP * PIECE || token_row(i, row) + 512u > SLOT) return false;
    }
    return true;
  }
};
// The row blocks that one XCD works on side by side (every eighth) walk K from eight places: in step they would all ask for the same 512 bytes
// of rows a power of two apart, which stand on a quarter of the L2's channels (10240 x 4096, 48 tokens: 32.1 -> 26.3 us; 32000 x 2048, 1 token 27.9 -> 24.2).
// The place follows from the row and K alone, whatever the tokens of the launch.  From eight chunks on and not in grouped or batched launches:
// those leave some shapes to the kernel above by their tokens, and a row is summed in one order in both (turn: 7, or 0).
__device__ __forceinline__ int first_chunk(int row, int chunks, int turn) { return ((row >> 7) & turn) * chunks / 8; }
static inline bool stream_narrow(int N, int token_tiles, int gz) { return (long)((N + 15) / 16) * token_tiles * gz <= 256; }

// whole chunks, 16-byte pieces from every row start, 32-bit offsets inside a workgroup's operands
static inline bool stream_ok(const void* x, const void* w, int N, int K, int epi, const LinExt& ext, int eb) {
  auto al = [eb](long n) { return n * eb % 16 == 0; };
  return (long)K * eb % 512 == 0 && al(ext.ldx) && al(ext.sx) && al(ext.sw) && al(ext.gs) && ((uintptr_t)x | (uintptr_t)w) % 16 == 0 &&
         ((epi_dual(epi) ? (long)N : 0L) + 64) * K * eb < (1L << 32) && (long)ext.ldx * 64 * eb < (1L << 32);
}

// Where the ring pays.  A workgroup fills three chunks before its first product and its LDS lets two of them on a unit, where the
// one-tile kernel has eight: with K of few chunks and more workgroups than units the latter is ahead, and a batch of prompts re-uses both
// operands, which its 64 x 64 tiles do and the ring's 32 rows do not.  us, one-tile kernel / ring, one MI355X, bf16: 32 x (512 x 256), 65 tokens
// 9.3 / 15.1; 32 x (128 x 512), 128 tokens 12.8 / 7.8 (256 workgroups), 200 15.6 / 15.9, 2000 66 / 114; 16384 x 1536, one token 10.3 / 11.2;
// 16384 x 256, 32 tokens 5.5 / 6.3; fp32 2048 x 256, 300 tokens 10.4 / 12.2, 32 x (256 x 512), 300 tokens 62 / 49.
static inline bool stream_pays(int T, int N, int K, int epi, int gz, int eb) {
  const long chunks = (long)K * eb / 512;
  const int rows = !epi_dual(epi) && T > 32 && !stream_narrow(N, (T + 63) / 64, gz) ? 32 : 16;
  const int tokens = T <= 16 ? 16 : T <= 32 ? 32 : T <= 48 ? 48 : 64;
  const long wgs = (long)((N + rows - 1) / rows) * ((T + tokens - 1) / tokens) * gz;
  if (wgs <= 256) return true;
  if (T <= 4 && eb == 2 && gz == 1) return chunks >= 8 || (epi_dual(epi) ? chunks > 2 || wgs <= 384 : wgs <= 512);
  if (T <= 64) return eb == 4 || chunks > 1 || wgs <= 384;
  return eb == 4 ? chunks > 2 : chunks > 1 && gz == 1;
}

// Streaming products of 33 to 64 tokens whose tokens stay in a workgroup's registers (seq_held.hip): where its 256 workgroups have more than one block of
// rows each (with one there is nothing to keep for), and K is 5 chunks (as long as the weights' ring) to 16, all that stay with a wave up to 48 tokens at 450 of
// 512 registers; of 64 tokens ten stay, the others are fetched again.  us, the streaming kernel / this, 33 / 48 / 64 tokens, gate/up 14336: K 1280 22.3 / 19.6,
// 22.3 / 19.0, 26.7 / 21.1; 2560 37.3 / 30.0, 39.7 / 31.7, 45.0 / 33.9; 3584 48.7 / 39.4, 49.2 / 40.8, 55.7 / 47.0; 12304 rows: 1280 13.0 / 12.6, 13.5 / 12.8, 15.7 / 14.2.
// Five chunks and a second block for an eighth of the workgroups or fewer: not (gate/up of 4112 and 4400, 48 tokens 9.5 / 10.4, 10.6 / 11.4; 5120 ahead).
constexpr int HELD_MIN = 5, HELD_MAX = 16;
static inline bool held_pays(int T, int N, int K, int epi) {
  const int one = epi_dual(epi) ? 256 : 512;
  return T > 32 && T <= 64 && (epi_plain(epi) || epi == EPI_CLAMP_GLU || epi == EPI_CAP) && K >= HELD_MIN * 256 && K <= HELD_MAX * 256 &&
         (N + 15) / 16 > (K == HELD_MIN * 256 ? one + one / 8 : one);
}
int held_stream(void* out, const void* x, const void* w, const void* bias, int T, int N, int K, int epi, float limit, float alpha, int dtype, hipStream_t st);
