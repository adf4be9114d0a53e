// Steps of 32 cached rows on their way through LDS, for the prompt attentions on the matrix pipe (seq_latent.hip, seq_battn.hip).
//
// A step's rows go from the paged cache to LDS by LDS-DMA, a KiB of consecutive 16-byte chunks an instruction: whole lines, no registers, and a step
// ahead of its use in the other of two buffers, so one barrier a step is enough.  (Through registers a thread fetched 16 bytes of a row of its own:
// every line was asked for four and more times, and behind two barriers.)  Chunk c of row r lies at place c ^ (r & XM) of the row, which the source
// address of a lane sees to: a fragment of 16 rows and a transposed one meet no bank conflict without padding.
// Keys are read as they lie (16 rows x 32 columns: the A operand of S^T = K Q^T).  Values are read with ds_read_b64_tr_b16: of 16 lanes, lane i
// names 8 bytes of row i / 4, columns 4 (i % 4) .., and receives column i of the four rows: the A operand of O^T += V^T P^T without a transposed copy
// (which took eight 2-byte LDS stores a chunk).
// The rows' places in the paged cache are looked up three steps ahead and stand in a table of two steps.
#pragma once
#include "gemm_tile.h"
#include "seq_decode.h"

typedef short s16x4_ __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_ lds_s16x4;

// 64 lanes x 16 B from an address of each lane's to LDS at ldsaddr + 16 * lane
__device__ __forceinline__ void rows_dma(const void* p, unsigned ldsaddr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(p), "s"(ldsaddr) : "memory", "m0");
}

template <int CHUNKS> struct RowTile {                          // rows of CHUNKS 16-byte chunks
  static constexpr int CH = (CHUNKS + 7) / 8 * 8, XM = CH % 16 == 0 ? 15 : 7, PIECES = CH / 2;
  static constexpr unsigned ROW = CH * 16u, BYTES = 32u * ROW;
};
// pkv_tok_row in two parts: the page asked for, and the row once it is there
struct RowAsked {
  int page, rest;
  __device__ __forceinline__ void ask(const UmbPagedKV& kv, int slot, int pos) {
    page = kv.pages[(long)slot * kv.max_pages + pos / kv.page];
    rest = pos % kv.page;
  }
  __device__ __forceinline__ unsigned row(const UmbPagedKV& kv, int g, int G) const { return ((unsigned)page * G + g) * kv.page + rest; }
};
// wave `wave` of NW fetches its pieces of a step; row_of(r): the place of the step's row r in units of rows, chunk_of(c): the chunk that stands at c,
// zeros where it is negative
static __device__ const u32x4 rows_zeros = {0u, 0u, 0u, 0u};
template <int CHUNKS, int NW, typename RowOf, typename ChunkOf>
__device__ __forceinline__ void rows_issue(const u16* base, long ld, unsigned lds, int wave, int lane, RowOf row_of, ChunkOf chunk_of) {
  typedef RowTile<CHUNKS> R;
  asm volatile("" : "+v"(lane));               // (or the places of every piece are kept in registers from step to step)
#pragma unroll
  for (int i = 0; i < (R::PIECES + NW - 1) / NW; ++i) {
    const int p = wave + NW * i, x = 64 * p + lane, r = x / R::CH, c = (x - r * R::CH) ^ (r & R::XM);
    if (i < R::PIECES / NW || p < R::PIECES) {
      const int ch = chunk_of(c);
      const u16* src = base + (long)row_of(r) * ld + 8 * ch;
      rows_dma(ch >= 0 ? src : reinterpret_cast<const u16*>(&rows_zeros), lds + (unsigned)p * 1024u);
    }
  }
}
// The same where every row fills its tile and a piece is whole rows: a piece's row and chunk are then a lane's own plus a constant, and an address is
// the look-up, a shift and an add.  (Put together from the piece's number they were 19 vector instructions a piece.)
template <int CHUNKS, int NW> struct RowLanes {
  typedef RowTile<CHUNKS> R;
  static constexpr bool OK = CHUNKS == R::CH && (R::CH & (R::CH - 1)) == 0 && R::CH <= 64 && R::PIECES % NW == 0;
  static constexpr int STEP = NW * 64 / R::CH;                  // rows from a wave's piece to its next
  const char* base;
  unsigned r0, c0;                                              // the first piece's row, and the place of its chunk in bytes
  __device__ __forceinline__ RowLanes(const u16* base, int wave, int lane)
      : base(reinterpret_cast<const char*>(base)), r0((unsigned)(wave * 64 + lane) / R::CH), c0(((unsigned)lane % R::CH ^ (r0 & R::XM)) * 16u) {}
  __device__ __forceinline__ void issue(const unsigned* rows, unsigned lds, int wave) const {
#pragma unroll
    for (int i = 0; i < R::PIECES / NW; ++i)
      rows_dma(base + (c0 ^ (unsigned)(STEP * i & R::XM) * 16u) + (size_t)rows[r0 + STEP * i] * R::ROW, lds + (unsigned)(wave + NW * i) * 1024u);
  }
};
// A operand of 16 rows (16 u ..) x 32 columns (chunks 4 s ..): lane (j, g) reads chunk 4 s + g of row j.  at_step: the addresses of a step's buffer, of
// which every read is one and a constant (opaque: put together from parts that do not change, each read's own would be kept over all steps)
template <int CHUNKS> struct RowKeys {
  typedef RowTile<CHUNKS> R;
  static constexpr int KINDS = (R::XM + 1) / 4;
  unsigned at, x, a[KINDS];
  __device__ __forceinline__ RowKeys(int j, int g) : at((unsigned)j * R::ROW), x((unsigned)(g ^ (j & R::XM)) * 16u) {}
  __device__ __forceinline__ void at_step(unsigned lds) {
#pragma unroll
    for (int i = 0; i < KINDS; ++i) {
      a[i] = lds + at + (x ^ (64u * i));
      asm volatile("" : "+v"(a[i]));
    }
  }
  __device__ __forceinline__ u32x4 operator()(int u, int s) const {
    return *reinterpret_cast<const lds_u32x4*>((size_t)(a[s % KINDS] + ((unsigned)(s / KINDS * KINDS * 64) + (unsigned)u * 16u * R::ROW)));
  }
};
// A operand of 16 columns (16 dt ..) x 32 keys: lane (j, g) receives column j of rows 4 g .. and 16 + 4 g ..
template <int CHUNKS> struct RowValues {
  typedef RowTile<CHUNKS> R;
  static constexpr int KINDS = (R::XM + 1) / 2;
  unsigned at, x, a[KINDS];
  __device__ __forceinline__ RowValues(int j, int g)
      : at((unsigned)(4 * g + (j >> 2)) * R::ROW), x((unsigned)(((j & 3) >> 1) ^ ((4 * g + (j >> 2)) & R::XM)) * 16u + (j & 1) * 8u) {}
  __device__ __forceinline__ void at_step(unsigned lds) {
#pragma unroll
    for (int i = 0; i < KINDS; ++i) {
      a[i] = lds + at + (x ^ (32u * i));
      asm volatile("" : "+v"(a[i]));
    }
  }
  __device__ __forceinline__ u32x4 operator()(int dt) const {
    const unsigned p = a[dt % KINDS] + (unsigned)(dt / KINDS * KINDS * 32);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>((size_t)p)));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>((size_t)(p + 16u * R::ROW))));
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
};
