// Gated linear attention: a [D][Dv] matrix state per (sequence, head), decayed per key channel and updated by an outer
// product at every token,
//     S_t = diag(alpha_t) S_(t-1) + k_t v_t^T        o_t = S_t^T q_t
// with alpha_t = sigmoid(W_a2 (W_a1 h_t) + b)^(1/tau) in (0, 1).  Everything here is fp32: the decay and its logarithm, the
// state, the products that enter it and the read-out.  The state lives in a slot array [slots][H][D][Dv] and is carried from
// step to step; a sequence whose first row is at position 0 starts from zero whatever its slot held before.
//
// scan kernel: one WAVE owns four value columns of one (sequence, head), or twice or four times as many (lin_scan_cols): lane (r = lane % 16, c = lane / 16)
// keeps NR consecutive rows (r NR ...) of column c in registers, so the update is register-local and the read-out sum over rows is a
// butterfly inside 16 lanes, and the order of every sum is fixed by (D) alone, in the kernels of single tokens too: how a sequence
// was cut into steps moves a token's output by the compiler's contractions at most (by the sums of the chunked form where a long stretch takes
// that).  The token loop is the only serial dimension; its inputs are independent of the recurrence and
// are staged ahead through LDS in chunks of 16 tokens.
#include "seq_common.h"
#include <type_traits>

// LOG: the decay's logarithm itself, as the chunked form reads it
template <typename P, bool LOG>
__global__ __launch_bounds__(256) void gla_decay_kernel(float* __restrict__ alpha, const float* __restrict__ proj, int ld,
                                                        int a_col, const typename El<P>::type* __restrict__ w_a2,
                                                        const typename El<P>::type* __restrict__ b_a2, int HD, int rank,
                                                        float inv_tau) {
  extern __shared__ float a_s[];
  const int t = blockIdx.x;
  for (int i = threadIdx.x; i < rank; i += 256) a_s[i] = proj[(long)t * ld + a_col + i];
  __syncthreads();
  for (int n = blockIdx.y * 256 + threadIdx.x; n < HD; n += gridDim.y * 256) {
    const typename El<P>::type* wr = w_a2 + (long)n * rank;
    float z = 0.f;
    for (int i = 0; i < rank; ++i) z += ldf<P>(wr + i) * a_s[i];
    if (b_a2) z += ldf<P>(b_a2 + n);
    const float la = log_sigmoidf_(z) * inv_tau;
    alpha[(long)t * HD + n] = LOG ? la : expf(la);
  }
}

constexpr int GLA_MAXR = 16;     // rows per lane: D <= 256
constexpr int GLA_TC = 16;       // tokens per staged chunk
constexpr int GLA_COLS = 16;     // value columns per workgroup (4 per wave)

// Workgroup = (sequence, head, 16 NC value columns), a lane NC of them 16 apart.  The token loop is serial, so its inputs must not
// cost a memory round trip per token: chunks of 16 tokens (alpha, k, q rows of the head and the 16 v columns) are staged
// through a double-buffered LDS tile -- the global loads of chunk c + 1 are in flight while chunk c is consumed from LDS.
// V4: D, Dv and the row stride of proj are multiples of 4 -> the staging moves 16-byte pieces (a quarter of the address
// arithmetic, which is what this issue-bound kernel spends its time on).
// Operand placement is general: q and k rows hold groups of D shared by `hpg` consecutive heads each (1: a group per head),
// and the decay is per key channel (alpha [T][H D]) or, with aph, one number per head (alpha [T][H]) that fills the staged
// row -- the state-space layers with a scalar decay per head run on the same kernel.
template <int NR, bool V4, int NC>
__global__ __launch_bounds__(256) void gla_scan_kernel(float* __restrict__ o, float* __restrict__ state,
                                                       const float* __restrict__ qp, int ldq, const float* __restrict__ kp,
                                                       int ldk, const float* __restrict__ vp, int ldv,
                                                       const float* __restrict__ alpha, int aph, int hpg,
                                                       const int* __restrict__ seq_slot, const int* __restrict__ seq_row0,
                                                       const int* __restrict__ seq_pos0, const int* __restrict__ seq_len, int H,
                                                       int D, int Dv, float qscale) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int VW = V4 ? 4 : 1;                        // floats per staged piece
  constexpr int WGC = GLA_COLS * NC;                    // the workgroup's columns; a thread's are 16 apart
  constexpr int STG = (3 * NR + NC + VW - 1) / VW;      // staged pieces per thread: TC (3 D + 16 NC) / 256 <= 3 NR + NC floats
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15;
  const int cbase = blockIdx.x * WGC, cl = wave * 4 + (lane >> 4), c = cbase + cl;
  const int h = blockIdx.y, b = blockIdx.z, hq = h / hpg;
  const int n = seq_len[b];
  if (n <= 0) return;
  const int slot = seq_slot[b], row0 = seq_row0[b];
  float* sp = state + (((long)slot * H + h) * D) * Dv + c;
  float S[NR][NC];
  const bool fresh = seq_pos0[b] == 0;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int d = r * NR + i;
#pragma unroll
    for (int x = 0; x < NC; ++x) S[i][x] = (!fresh && c + 16 * x < Dv && d < D) ? sp[(long)d * Dv + 16 * x] : 0.f;
  }
  const int HD = H * D, rowlen = 3 * D + WGC, chunk = GLA_TC * rowlen;
  const int nch = (n + GLA_TC - 1) / GLA_TC;
  typedef typename std::conditional<V4, f32x4, float>::type piece;
  piece stage[STG];
  const int rowp = rowlen / VW, chunkp = chunk / VW;    // in pieces
  // chunk ch -> registers.  Every load is unconditional and lands on a valid address (indices are clamped): loads that sit in
  // divergent branches would each wait for their own round trip.  What a clamped load brings is never used: tokens past the
  // sequence are not consumed, columns past Dv are not written, indices past the chunk are not stashed.
  const int tt0 = tid / rowp, ci0 = (tid - tt0 * rowp) * VW;
  auto fetch = [&](int ch) {
    int tt = tt0, ci = ci0;                             // (token, column) of staged piece e * 256 + tid, kept incrementally
#pragma unroll
    for (int e = 0; e < STG; ++e) {
      if (e) {
        ci += 256 * VW;
        while (ci >= rowlen) { ci -= rowlen; ++tt; }
        if (tt >= GLA_TC) { tt = GLA_TC - 1; ci = rowlen - VW; }     // past the chunk: any valid address
      }
      int t = ch * GLA_TC + tt;
      t = t < n ? t : n - 1;
      const long row = row0 + t;
      int vc = cbase + ci - 3 * D;
      vc = vc + VW <= Dv ? vc : Dv - VW;
      const bool is_a = ci < D;
      const float* src = (is_a && !aph) ? alpha + row * HD + (long)h * D + ci
                       : ci < 2 * D ? kp + row * ldk + (long)hq * D + (is_a ? ci : ci - D)
                       : ci < 3 * D ? qp + row * ldq + (long)hq * D + (ci - 2 * D)
                                    : vp + row * ldv + (long)h * Dv + vc;
      stage[e] = *reinterpret_cast<const piece*>(src);
      if (aph) {                                        // uniform: one decay per head fills the alpha part of the row
        const float a = alpha[row * H + h];
        if (is_a) {
          if constexpr (V4) stage[e] = piece{a, a, a, a};
          else stage[e] = a;
        }
      }
    }
  };
  auto stash = [&](float* buf) {
#pragma unroll
    for (int e = 0; e < STG; ++e) {
      const int idx = e * 256 + tid;
      if (idx < chunkp) reinterpret_cast<piece*>(buf)[idx] = stage[e];
    }
  };
  fetch(0);
  stash(lds);
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const float* buf = lds + (ch & 1) * chunk;
    if (ch + 1 < nch) fetch(ch + 1);
    const int cnt = n - ch * GLA_TC < GLA_TC ? n - ch * GLA_TC : GLA_TC;
    float pt[NC][GLA_TC];                               // this lane's share (its rows) of every token's read-out
#pragma unroll
    for (int tt = 0; tt < GLA_TC; ++tt) {
      float acc[NC] = {};
      if (tt < cnt) {
        const float* row = buf + tt * rowlen;
        float v[NC];
#pragma unroll
        for (int x = 0; x < NC; ++x) v[x] = row[3 * D + cl + 16 * x];
        float al[NR], kk[NR], qq[NR];
        bool got = false;
        if constexpr (NR % 4 == 0) {
          if ((D & 3) == 0) {                           // 16-byte LDS reads of the lane's NR consecutive rows
#pragma unroll
            for (int i = 0; i < NR; i += 4) {
              const f32x4 a4 = *reinterpret_cast<const f32x4*>(row + r * NR + i);
              const f32x4 k4 = *reinterpret_cast<const f32x4*>(row + D + r * NR + i);
              const f32x4 q4 = *reinterpret_cast<const f32x4*>(row + 2 * D + r * NR + i);
#pragma unroll
              for (int e = 0; e < 4; ++e) { al[i + e] = a4[e]; kk[i + e] = k4[e]; qq[i + e] = q4[e]; }
            }
            got = true;
          }
        }
        if (!got) {
#pragma unroll
          for (int i = 0; i < NR; ++i) {
            const int d = r * NR + i;
            al[i] = row[d]; kk[i] = row[D + d]; qq[i] = row[2 * D + d];
          }
        }
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          if (r * NR + i < D) {
#pragma unroll
            for (int x = 0; x < NC; ++x) {
              S[i][x] = al[i] * S[i][x] + kk[i] * v[x];
              acc[x] += S[i][x] * qq[i];
            }
          }
        }
      }
#pragma unroll
      for (int x = 0; x < NC; ++x) pt[x][tt] = acc[x];
    }
    // sum over the 16 row lanes, all 16 tokens at once: a transposing butterfly (15 exchanges instead of 64).  At the step with
    // mask m a lane keeps the half of its values whose token bit m equals its own lane bit and hands the other half to its
    // partner; lane r ends up with the whole sum of token r.  Every token's sum has the same tree (pairs by 8, 4, 2, 1).
#pragma unroll
    for (int x = 0; x < NC; ++x) {
      float p8[8], p4[4], p2[2];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool up = r & 8;
        p8[j] = (up ? pt[x][j + 8] : pt[x][j]) + __shfl_xor(up ? pt[x][j] : pt[x][j + 8], 8, 64);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool up = r & 4;
        p4[j] = (up ? p8[j + 4] : p8[j]) + __shfl_xor(up ? p8[j] : p8[j + 4], 4, 64);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bool up = r & 2;
        p2[j] = (up ? p4[j + 2] : p4[j]) + __shfl_xor(up ? p4[j] : p4[j + 2], 2, 64);
      }
      const bool up1 = r & 1;
      const float mine = ((up1 ? p2[1] : p2[0]) + __shfl_xor(up1 ? p2[0] : p2[1], 1, 64)) * qscale;
      if (r < cnt && c + 16 * x < Dv) o[(long)(row0 + ch * GLA_TC + r) * (H * Dv) + (long)h * Dv + c + 16 * x] = mine;
    }
    if (ch + 1 < nch) stash(lds + ((ch + 1) & 1) * chunk);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int d = r * NR + i;
#pragma unroll
    for (int x = 0; x < NC; ++x)
      if (d < D && c + 16 * x < Dv) sp[(long)d * Dv + 16 * x] = S[i][x];
  }
}

template <typename P>
__global__ __launch_bounds__(256) void gla_gate_kernel(typename El<P>::type* __restrict__ out, const float* __restrict__ o,
                                                       const float* __restrict__ proj, int ld, int g_col,
                                                       const typename El<P>::type* __restrict__ w, int T, int H, int Dv, float eps) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long th = (long)blockIdx.x * 4 + wave;           // (token, head)
  if (th >= (long)T * H) return;
  const int t = (int)(th / H), h = (int)(th % H);
  const float* orow = o + (long)t * H * Dv + (long)h * Dv;
  float ss = 0.f;
  for (int i = lane; i < Dv; i += 64) { const float v = orow[i]; ss += v * v; }
  ss = wave_sum(ss);
  const float f = 1.f / sqrtf(ss / (float)Dv + eps);
  const float* gr = proj + (long)t * ld + g_col + (long)h * Dv;
  for (int i = lane; i < Dv; i += 64)
    stf<P>(out + (long)t * H * Dv + (long)h * Dv + i, orow[i] * f * ldf<P>(w + i) * siluf_(gr[i]));
}

template <bool LOG>
static int gla_decay_launch(float* alpha, const float* proj, int ld, int a_col, const void* w_a2, const void* b_a2, int T, int HD, int rank,
                            float tau, int dtype, hipStream_t st) {
  if (T < 1 || HD < 1 || rank < 1 || rank > 8192 || !(tau > 0.f) || !alpha || !proj || !w_a2) return UMB_EINVAL;
  const int gy = (HD + 255) / 256 > 64 ? 64 : (HD + 255) / 256;
  DISPATCH_SEQ_DTYPE(dtype, {
    typedef typename El<P>::type E;
    hipLaunchKernelGGL((gla_decay_kernel<P, LOG>), dim3(T, gy), dim3(256), rank * sizeof(float), st, alpha, proj, ld, a_col,
                       (const E*)w_a2, (const E*)b_a2, HD, rank, 1.f / tau);
  })
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_gla_decay(float* alpha, const float* proj, int ld, int a_col, const void* w_a2, const void* b_a2, int T, int HD,
                             int rank, float tau, int dtype, hipStream_t st) {
  return gla_decay_launch<false>(alpha, proj, ld, a_col, w_a2, b_a2, T, HD, rank, tau, dtype, st);
}

extern "C" int umb_gla_decay_log(float* log_alpha, const float* proj, int ld, int a_col, const void* w_a2, const void* b_a2, int T, int HD,
                                 int rank, float tau, int dtype, hipStream_t st) {
  return gla_decay_launch<true>(log_alpha, proj, ld, a_col, w_a2, b_a2, T, HD, rank, tau, dtype, st);
}

extern "C" int umb_lin_scan_columns(int T, int max_len, int H, int D, int Dv) {
  return T < 1 || H < 1 || D < 1 || D > 16 * GLA_MAXR || Dv < 1 ? UMB_EINVAL : lin_scan_cols(T, max_len, H, D, Dv);
}

extern "C" int umb_lin_scan_rows(float* o, float* state, const float* q, int ldq, const float* k, int ldk, const float* v, int ldv,
                                 const float* alpha, int alpha_per_head, int qk_heads, const int* seq_slot, const int* seq_row0,
                                 const int* seq_pos0, const int* seq_len, int T, int B, int max_len, int H, int D, int Dv, float qscale,
                                 hipStream_t st) {
  if (B < 1 || H < 1 || D < 1 || D > 16 * GLA_MAXR || Dv < 1 || qk_heads < 1 || H % qk_heads || !o || !state ||
      !q || !k || !v || !alpha || ldq < qk_heads * D || ldk < qk_heads * D || ldv < H * Dv)
    return UMB_EINVAL;
  const int nr = (D + 15) / 16, aph = alpha_per_head ? 1 : 0, hpg = H / qk_heads;
  const bool v4 = D % 4 == 0 && Dv % 4 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 &&
                  ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (aph ? 0 : (uintptr_t)alpha)) % 16 == 0;
  const int nc = v4 ? lin_scan_cols(T, max_len, H, D, Dv) : 1;
  const dim3 grid((Dv + GLA_COLS * nc - 1) / (GLA_COLS * nc), H, B);
#define GLA_SCAN_LAUNCH(NR, V4, NC)                                                                                       \
  do {                                                                                                                    \
    const size_t lds = 2 * (size_t)GLA_TC * (3 * D + GLA_COLS * NC) * sizeof(float);                                      \
    if (ensure_dynamic_lds<gla_scan_kernel<NR, V4, NC>>(lds) != UMB_OK) return UMB_EHIP;                                  \
    hipLaunchKernelGGL((gla_scan_kernel<NR, V4, NC>), grid, dim3(256), lds, st, o, state, q, ldq, k, ldk, v, ldv, alpha, aph, \
                       hpg, seq_slot, seq_row0, seq_pos0, seq_len, H, D, Dv, qscale);                                     \
  } while (0)
#define GLA_SCAN_CASE(NR)                                                                                                 \
  case NR:                                                                                                                \
    if (v4) GLA_SCAN_LAUNCH(NR, true, 1); else GLA_SCAN_LAUNCH(NR, false, 1);                                             \
    break;
#define GLA_SCAN_WIDE(NR)                                                                                                 \
  case NR:                                                                                                                \
    if (nc == 4) GLA_SCAN_LAUNCH(NR, true, 4); else GLA_SCAN_LAUNCH(NR, true, 2);                                         \
    break;
  if (nc > 1) {
    switch (nr) {
      GLA_SCAN_WIDE(4) GLA_SCAN_WIDE(8) GLA_SCAN_WIDE(12) GLA_SCAN_WIDE(16)
    }
  } else {
    switch (nr) {
      GLA_SCAN_CASE(1) GLA_SCAN_CASE(2) GLA_SCAN_CASE(3) GLA_SCAN_CASE(4) GLA_SCAN_CASE(5) GLA_SCAN_CASE(6) GLA_SCAN_CASE(7)
      GLA_SCAN_CASE(8) GLA_SCAN_CASE(9) GLA_SCAN_CASE(10) GLA_SCAN_CASE(11) GLA_SCAN_CASE(12) GLA_SCAN_CASE(13)
      GLA_SCAN_CASE(14) GLA_SCAN_CASE(15) GLA_SCAN_CASE(16)
      default: return UMB_EINVAL;
    }
  }
#undef GLA_SCAN_CASE
#undef GLA_SCAN_WIDE
#undef GLA_SCAN_LAUNCH
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_lin_scan(float* o, float* state, const float* q, int ldq, const float* k, int ldk, const float* v, int ldv,
                            const float* alpha, int alpha_per_head, int qk_heads, const int* seq_slot, const int* seq_row0,
                            const int* seq_pos0, const int* seq_len, int B, int H, int D, int Dv, float qscale, hipStream_t st) {
  return umb_lin_scan_rows(o, state, q, ldq, k, ldk, v, ldv, alpha, alpha_per_head, qk_heads, seq_slot, seq_row0, seq_pos0, seq_len, 1, B, 0, H, D, Dv,
                           qscale, st);
}

extern "C" int umb_gla_scan(float* o, float* state, const float* proj, int ld, const float* alpha, const int* seq_slot,
                            const int* seq_row0, const int* seq_pos0, const int* seq_len, int B, int H, int D, int Dv,
                            float qscale, hipStream_t st) {
  if (!proj || H < 1 || D < 1 || Dv < 1 || ld < 2 * H * D + H * Dv) return UMB_EINVAL;
  return umb_lin_scan(o, state, proj, ld, proj + (long)H * D, ld, proj + 2L * H * D, ld, alpha, 0, H, seq_slot, seq_row0, seq_pos0,
                      seq_len, B, H, D, Dv, qscale, st);
}

extern "C" int umb_gla_gate(void* out, const float* o, const float* proj, int ld, int g_col, const void* w, int T, int H, int Dv,
                            float eps, int dtype, hipStream_t st) {
  if (T < 1 || H < 1 || Dv < 1 || !out || !o || !proj || !w) return UMB_EINVAL;
  const long th = (long)T * H;
  DISPATCH_SEQ_DTYPE(dtype, {
    typedef typename El<P>::type E;
    hipLaunchKernelGGL(gla_gate_kernel<P>, dim3((unsigned)((th + 3) / 4)), dim3(256), 0, st, (E*)out, o, proj, ld, g_col,
                       (const E*)w, T, H, Dv, eps);
  })
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// ---- one token per sequence: the state is read and written once, nothing else is large (16 requests x 16 heads x 128 x 256: 67 MB).
// Workgroup = (64 value columns, head, token): thread (column quad tid % 16, row group r = tid / 16) keeps rows r nr .. of its four
// columns, all loads in flight at once; the read-out sums rows as the scan does (nr in order, then groups by 8, 4, 2, 1).
// The scan kernel stages sixteen tokens' operands for the one: 46 us for those 67 MB, 13.6 here (4.9 TB/s); 8 heads x 128 x 256, one request
// 10.6 -> 5.4.
template <int RMAX>
__global__ __launch_bounds__(256) void lin_step_kernel(float* __restrict__ o, float* __restrict__ state, const float* __restrict__ qp, int ldq,
                                                       const float* __restrict__ kp, int ldk, const float* __restrict__ vp, int ldv,
                                                       const float* __restrict__ alpha, int aph, int hpg, const int* __restrict__ pos,
                                                       const int* __restrict__ slot, int H, int D, int Dv, float qscale) {
  __shared__ __attribute__((aligned(16))) float rowv[3][16 * GLA_MAXR];          // alpha, k, q of the head
  __shared__ __attribute__((aligned(16))) float red[16][64];
  const int t = blockIdx.z, h = blockIdx.y, hq = h / hpg, nr = (D + 15) / 16;
  const int cq = threadIdx.x & 15, r = threadIdx.x >> 4, c = blockIdx.x * 64 + 4 * cq;
  const bool c_ok = c < Dv;
  float* sp = state + (((long)slot[t] * H + h) * D) * Dv + (c_ok ? c : 0);
  f32x4 S[RMAX];
#pragma unroll
  for (int i = 0; i < RMAX; ++i) {
    const int d = r * nr + (i < nr ? i : nr - 1);
    S[i] = *reinterpret_cast<const f32x4*>(sp + (long)(d < D ? d : D - 1) * Dv);
  }
  const f32x4 v = *reinterpret_cast<const f32x4*>(vp + (long)t * ldv + (long)h * Dv + (c_ok ? c : 0));
  const int d0 = threadIdx.x;
  if (d0 < D) {
    rowv[0][d0] = aph ? alpha[(long)t * H + h] : alpha[(long)t * H * D + (long)h * D + d0];
    rowv[1][d0] = kp[(long)t * ldk + (long)hq * D + d0];
    rowv[2][d0] = qp[(long)t * ldq + (long)hq * D + d0];
  }
  const bool fresh = pos[t] == 0;
  __syncthreads();
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RMAX; ++i) {
    const int d = r * nr + i;
    if (i < nr && d < D) {
      const float al = rowv[0][d], kk = rowv[1][d], qq = rowv[2][d];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        S[i][e] = al * (fresh ? 0.f : S[i][e]) + kk * v[e];
        acc[e] += S[i][e] * qq;
      }
      if (c_ok) *reinterpret_cast<f32x4*>(sp + (long)d * Dv) = S[i];
    }
  }
  *reinterpret_cast<f32x4*>(&red[r][4 * cq]) = acc;
  __syncthreads();
  const int cc = threadIdx.x;
  if (cc < 64 && blockIdx.x * 64 + cc < Dv) {
    float p[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) p[i] = red[i][cc];
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1)
#pragma unroll
      for (int i = 0; i < m; ++i) p[i] += p[i + m];
    o[(long)t * (H * Dv) + (long)h * Dv + blockIdx.x * 64 + cc] = p[0] * qscale;
  }
}

extern "C" int umb_lin_step(float* o, float* state, const float* q, int ldq, const float* k, int ldk, const float* v, int ldv,
                            const float* alpha, int alpha_per_head, int qk_heads, const int* pos, const int* slot, int T, int H, int D, int Dv,
                            float qscale, hipStream_t st) {
  if (T < 1 || T > 65535 || H < 1 || H > 65535 || D < 1 || D > 16 * GLA_MAXR || Dv < 1 || Dv % 4 || qk_heads < 1 || H % qk_heads || !o || !state ||
      !q || !k || !v || !alpha || !pos || !slot || ldq < qk_heads * D || ldk < qk_heads * D || ldv < H * Dv || ldv % 4 ||
      ((uintptr_t)v | (uintptr_t)state) % 16)
    return UMB_EINVAL;
  const dim3 grid((Dv + 63) / 64, H, T);
  const int nr = (D + 15) / 16, aph = alpha_per_head ? 1 : 0, hpg = H / qk_heads;
#define LIN_STEP(R) \
  hipLaunchKernelGGL(lin_step_kernel<R>, grid, dim3(256), 0, st, o, state, q, ldq, k, ldk, v, ldv, alpha, aph, hpg, pos, slot, H, D, Dv, qscale)
  if (nr <= 2) LIN_STEP(2);
  else if (nr <= 4) LIN_STEP(4);
  else if (nr <= 8) LIN_STEP(8);
  else LIN_STEP(16);
#undef LIN_STEP
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// ---- the same with what stands around it in gated linear attention: the decays from the rank-`rank` product in front, the head's norm and its gate behind.
// Workgroup = (head, token): CG groups of 256 threads, each 64 value columns as above.  As three launches decay, step and gate took 4.9 + 11.4 + 4.8 us for 16
// requests x 16 heads x 128 x 256, here 14.4; one request, 8 heads 3.5 + 5.5 + 4.5, here 8.7.
template <typename P, int RMAX, int CG>
__global__ __launch_bounds__(256 * CG) void gla_step_kernel(typename El<P>::type* __restrict__ out, float* __restrict__ state, const float* __restrict__ proj, int ld,
                                                            const typename El<P>::type* __restrict__ w_a2, const typename El<P>::type* __restrict__ b_a2,
                                                            const typename El<P>::type* __restrict__ w_norm, const int* __restrict__ pos,
                                                            const int* __restrict__ slot, int H, int D, int Dv, int rank, float inv_tau, float qscale, float eps) {
  __shared__ __attribute__((aligned(16))) float rowv[3][16 * GLA_MAXR];          // alpha, k, q of the head
  __shared__ __attribute__((aligned(16))) float red[CG][16][64];
  __shared__ float squares[CG];
  const int h = blockIdx.x, t = blockIdx.y, nr = (D + 15) / 16, HD = H * D;
  const int cg = threadIdx.x >> 8, in = threadIdx.x & 255, cq = in & 15, r = in >> 4, c = cg * 64 + 4 * cq;
  const bool c_ok = c < Dv;
  const float* row = proj + (long)t * ld;
  float* sp = state + (((long)slot[t] * H + h) * D) * Dv + (c_ok ? c : 0);
  f32x4 S[RMAX];
#pragma unroll
  for (int i = 0; i < RMAX; ++i) {
    const int d = r * nr + (i < nr ? i : nr - 1);
    S[i] = *reinterpret_cast<const f32x4*>(sp + (long)(d < D ? d : D - 1) * Dv);
  }
  typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
  const f32x4 v = *reinterpret_cast<const quad*>(row + 2L * HD + (long)h * Dv + (c_ok ? c : 0));
  const int d0 = threadIdx.x;
  if (d0 < D) {
    const typename El<P>::type* wr = w_a2 + ((long)h * D + d0) * rank;
    const float* a = row + 2L * HD + 2L * H * Dv;
    float z = 0.f;
    for (int i0 = 0; i0 < rank; i0 += 8) {                 // in order, eight of them on their way at a time
      float wv[8], av[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        wv[i] = ldf<P>(wr + min(i0 + i, rank - 1));
        av[i] = a[min(i0 + i, rank - 1)];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i0 + i < rank) z += wv[i] * av[i];
    }
    if (b_a2) z += ldf<P>(b_a2 + (long)h * D + d0);
    rowv[0][d0] = expf(log_sigmoidf_(z) * inv_tau);
    rowv[1][d0] = row[HD + (long)h * D + d0];
    rowv[2][d0] = row[(long)h * D + d0];
  }
  const bool fresh = pos[t] == 0;
  __syncthreads();
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RMAX; ++i) {
    const int d = r * nr + i;
    if (i < nr && d < D) {
      const float al = rowv[0][d], kk = rowv[1][d], qq = rowv[2][d];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        S[i][e] = al * (fresh ? 0.f : S[i][e]) + kk * v[e];
        acc[e] += S[i][e] * qq;
      }
      if (c_ok) *reinterpret_cast<f32x4*>(sp + (long)d * Dv) = S[i];
    }
  }
  *reinterpret_cast<f32x4*>(&red[cg][r][4 * cq]) = acc;
  __syncthreads();
  const int cc = cg * 64 + in;
  const bool mine = in < 64 && cc < Dv;
  float o = 0.f;
  if (mine) {
    float p[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) p[i] = red[cg][i][in];
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1)
#pragma unroll
      for (int i = 0; i < m; ++i) p[i] += p[i + m];
    o = p[0] * qscale;
  }
  const float ss = wave_sum(o * o);
  if (in == 0) squares[cg] = ss;
  __syncthreads();
  if (!mine) return;
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < CG; ++i) total += squares[i];
  const float f = 1.f / sqrtf(total / (float)Dv + eps);
  stf<P>(out + ((long)t * H + h) * Dv + cc, o * f * ldf<P>(w_norm + cc) * siluf_(row[2L * HD + (long)H * Dv + (long)h * Dv + cc]));
}

extern "C" int umb_gla_step(void* out, float* state, const float* proj, int ld, const void* w_a2, const void* b_a2, const void* w_norm, const int* pos,
                            const int* slot, int T, int H, int D, int Dv, int rank, float tau, float qscale, float eps, int dtype, hipStream_t st) {
  if (T < 1 || T > 65535 || H < 1 || D < 1 || D > 16 * GLA_MAXR || Dv < 4 || Dv % 4 || Dv > 256 || rank < 1 || rank > 8192 || !(tau > 0.f) || !out || !state || !proj ||
      !w_a2 || !w_norm || !pos || !slot || (long)ld < 2L * H * D + 2L * H * Dv + rank || (uintptr_t)state % 16)
    return UMB_EINVAL;
  const int nr = (D + 15) / 16;
#define GLA_STEP(R, CG)                                                                                                                       \
  hipLaunchKernelGGL((gla_step_kernel<P, R, CG>), dim3(H, T), dim3(256 * CG), 0, st, (E*)out, state, proj, ld, (const E*)w_a2, (const E*)b_a2, \
                     (const E*)w_norm, pos, slot, H, D, Dv, rank, 1.f / tau, qscale, eps)
#define GLA_STEP_C(R) do { if (Dv <= 64) GLA_STEP(R, 1); else if (Dv <= 128) GLA_STEP(R, 2); else GLA_STEP(R, 4); } while (0)
  DISPATCH_SEQ_DTYPE(dtype, {
    typedef typename El<P>::type E;
    if (nr <= 4) GLA_STEP_C(4);
    else if (nr <= 8) GLA_STEP_C(8);
    else GLA_STEP_C(16);
  })
#undef GLA_STEP_C
#undef GLA_STEP
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

// ---- the recurrence in chunks of 64 tokens, for stretches of many.  With one decay per key CHANNEL, c_t = sum of the channel's
// log decays over the chunk up to and including token t:
//     S_end = e^(c_64) S_start + sum_s (e^(c_64 - c_s) k_s) v_s^T        o_t = (e^(c_t) q_t)^T S_start + sum_{s <= t} A_ts v_s
//     A_ts  = sum_d q_td k_sd e^(c_td - c_sd)
// All exponents are of non-positive numbers.  A's 16 x 16 blocks below the diagonal split the exponent at the start r of the row
// block, (e^(c_t - r) q_t) . (e^(r - c_s) k_s), a matrix product; in the diagonal blocks the split would need e^(+): there every
// pair of tokens and channel takes its own exponential.  Four launches, all but the second over (column slice, chunk, head, sequence):
//   prep   c (prefix sums in double and base 2, kept as blocks' starts and offsets inside a block in two 32-bit parts), A, e^(c_t) q_t,
//          e^(c_64 - c_s) k_s
//   state  every chunk's sum from a zero state        pass   chunks in order: sums become start states, the slot the final one
//   out    A v + (e^c q)^T S_start
// fp32 throughout, products on the fp32 matrix pipe.  2048 tokens, 8 heads x 128 x 256 on one MI355X: 670 us token by token (a serial
// loop on 512 waves) -> 92; 192 tokens 66 -> 45.  D and Dv multiples of 16, D <= 128 (the chunk's q, k and offsets fill the LDS).
// Values that are not finite stay where the recurrence has them: a log decay below GC_LA (a decay of zero in fp32, -inf included) is taken
// as that; later tokens of a block meet an infinite value with weight zero, so such a block is summed token by token.
constexpr int GC_Q = 64;
constexpr float GC_LA = -128.f;
// An offset inside a block as r + l / ln 2: r a multiple of 2^-12 (below 4096: 24 bits, so a difference of two is exact), l small.
// e^(difference) = 2^dr (1 + dl) is then good to 2^-22 however large it is, where an exponent x rounded to 32 bits costs x 2^-24.  Relative error
// of the weights inside a block, largest / root mean square in 2^-24, decays of 4 a token: 2.1 / 0.58; with the rounded exponent 149 / 19;
// token by token 7.9 / 1.3.
constexpr double GC_LOG2E = 1.4426950408889634, GC_LN2 = 0.6931471805599453;
__device__ __forceinline__ float gla_exp(float r, float l) {
  const float v = __builtin_amdgcn_exp2f(r);
  return fmaf(v, l, v);
}
__device__ __forceinline__ float gla_exp(double c) {        // 2^c
  const float r = (float)c;
  return gla_exp(r, (float)((c - (double)r) * GC_LN2));
}

struct GlaChunk {
  const float *q, *k, *v, *la;             // rows of proj at the q, k, v columns; la [T][H D]
  int ld, H, D, Dv;
  const int *seq_slot, *seq_row0, *seq_pos0, *seq_len;
  float *qt, *kh, *m, *sc, *ac;            // [T][H D] twice, [T][H][64], [chunks][H][D][Dv], [chunks][H][D]
  float qscale;
  // chunks of the sequences before b
  __device__ __forceinline__ int first(int b) const {
    int n = 0;
    for (int i = 0; i < b; ++i) n += (seq_len[i] + GC_Q - 1) / GC_Q;
    return n;
  }
};

__device__ __forceinline__ f32x4 gla_mma(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// grid (chunks, heads, sequences).  One workgroup fills a CU's LDS: 1024 threads, 256 for each diagonal block, whose exponentials are most
// of the work (256 threads: 40 us for one chunk as for 256 of them)
__global__ __launch_bounds__(1024) void gla_chunk_prep_kernel(GlaChunk a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int b = blockIdx.z, h = blockIdx.y, t0 = blockIdx.x * GC_Q, len = a.seq_len[b];
  if (t0 >= len) return;
  const int cnt = len - t0 < GC_Q ? len - t0 : GC_Q, D = a.D, LD = D + 4, HD = a.H * D;
  const long row0 = (long)a.seq_row0[b] + t0;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
  double* blk = reinterpret_cast<double*>(sm);   // [5][128]: c at the starts of the four blocks, and at the chunk's end
  float* rs = sm + 2 * 5 * 128;                  // [64][LD]: c_t less the start of t's block: r ..
  float* rl = rs + GC_Q * LD;                    // [64][LD]: .. and l
  float* qs = rl + GC_Q * LD;                    // [64][LD]
  float* ks = qs + GC_Q * LD;                    // [64][LD]
  if (tid < 512 && (tid & 127) < D) {            // (channel, block): the block's running sums
    const int d = tid & 127, u = tid >> 7;
    float l[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = 16 * u + i;
      const float la = a.la[(row0 + (t < cnt ? t : cnt - 1)) * HD + (long)h * D + d];
      l[i] = la < GC_LA ? GC_LA : la;            // a NaN stays one
    }
    double run = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = 16 * u + i;
      run += t < cnt ? GC_LOG2E * (double)l[i] : 0.0;
      const double r = rint(run * 4096.0) / 4096.0;
      rs[t * LD + d] = (float)r;
      rl[t * LD + d] = (float)((run - r) * GC_LN2);
    }
    blk[(u + 1) * 128 + d] = run;                // the block's own sum for now
  }
  const int dq = D >> 2;
  for (int x = tid; x < GC_Q * dq; x += 1024) {
    const int t = x / dq, d = (x - t * dq) * 4;
    f32x4 qv = f32x4{0.f, 0.f, 0.f, 0.f}, kv = qv;
    if (t < cnt) {
      qv = *reinterpret_cast<const f32x4*>(a.q + (row0 + t) * a.ld + (long)h * D + d);
      kv = *reinterpret_cast<const f32x4*>(a.k + (row0 + t) * a.ld + (long)h * D + d);
    }
    *reinterpret_cast<f32x4*>(qs + t * LD + d) = qv;
    *reinterpret_cast<f32x4*>(ks + t * LD + d) = kv;
  }
  __syncthreads();
  const int nc = a.first(b) + blockIdx.x;
  if (tid < D) {
    double run = 0.0;
    blk[tid] = 0.0;
#pragma unroll
    for (int i = 1; i <= 4; ++i) {
      run += blk[i * 128 + tid];
      blk[i * 128 + tid] = run;
    }
    a.ac[((long)nc * a.H + h) * D + tid] = gla_exp(run);
  }
  __syncthreads();
  for (int x = tid; x < GC_Q * dq; x += 1024) {   // what the other launches read: decayed from the chunk's start, to its end
    const int t = x / dq, d = (x - t * dq) * 4;
    if (t >= cnt) continue;
    f32x4 qv = *reinterpret_cast<const f32x4*>(qs + t * LD + d), kv = *reinterpret_cast<const f32x4*>(ks + t * LD + d);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double c = blk[(t >> 4) * 128 + d + e] + ((double)rs[t * LD + d + e] + GC_LOG2E * (double)rl[t * LD + d + e]);
      qv[e] *= gla_exp(c);
      kv[e] *= gla_exp(blk[4 * 128 + d + e] - c);
    }
    *reinterpret_cast<f32x4*>(a.qt + (row0 + t) * HD + (long)h * D + d) = qv;
    *reinterpret_cast<f32x4*>(a.kh + (row0 + t) * HD + (long)h * D + d) = kv;
  }
  // diagonal block tid / 256: thread (row, column)
  const int tr = (tid >> 4) & 15, ts = tid & 15;
  {
    const int t = 16 * (tid >> 8) + tr, s = 16 * (tid >> 8) + ts;
    float acc = 0.f;
    if (ts <= tr && t < cnt) {
      for (int d = 0; d < D; d += 4) {
        const f32x4 q4 = *reinterpret_cast<const f32x4*>(qs + t * LD + d), k4 = *reinterpret_cast<const f32x4*>(ks + s * LD + d);
        const f32x4 rt = *reinterpret_cast<const f32x4*>(rs + t * LD + d), r4 = *reinterpret_cast<const f32x4*>(rs + s * LD + d);
        const f32x4 lt = *reinterpret_cast<const f32x4*>(rl + t * LD + d), l4 = *reinterpret_cast<const f32x4*>(rl + s * LD + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc += q4[e] * k4[e] * gla_exp(rt[e] - r4[e], lt[e] - l4[e]);
      }
    }
    if (t < cnt) a.m[((row0 + t) * a.H + h) * 64 + s] = acc;
  }
  // the six blocks below the diagonal: row block rb, column block cb
  if (wave < 6) {
    const int id = wave;
    const int rb = id < 1 ? 1 : (id < 3 ? 2 : 3), cb = id - rb * (rb - 1) / 2;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const int t = 16 * rb + j, s = 16 * cb + j;
    for (int k0 = 4 * g; k0 < D; k0 += 16) {
      f32x4 x = *reinterpret_cast<const f32x4*>(qs + t * LD + k0), y = *reinterpret_cast<const f32x4*>(ks + s * LD + k0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] *= gla_exp(rs[t * LD + k0 + e], rl[t * LD + k0 + e]);
        y[e] *= gla_exp(blk[rb * 128 + k0 + e] - (blk[cb * 128 + k0 + e] + ((double)rs[s * LD + k0 + e] + GC_LOG2E * (double)rl[s * LD + k0 + e])));
      }
      acc = gla_mma(x, y, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tt = 16 * rb + 4 * g + r;
      if (tt < cnt) a.m[((row0 + tt) * a.H + h) * 64 + 16 * cb + j] = acc[r];
    }
  }
}

// grid (64-column slices, chunks, sequences x heads): wave w the row tiles w, w + 4 of the state, four column tiles
__global__ __launch_bounds__(256) void gla_chunk_state_kernel(GlaChunk a) {
  const int b = blockIdx.z / a.H, h = blockIdx.z % a.H, t0 = blockIdx.y * GC_Q, len = a.seq_len[b];
  if (t0 >= len) return;
  const int cnt = len - t0 < GC_Q ? len - t0 : GC_Q, D = a.D, Dv = a.Dv, HD = a.H * D;
  const long row0 = (long)a.seq_row0[b] + t0;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, p0 = blockIdx.x * 64;
  f32x4 acc[2][4];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k0 = 0; k0 < GC_Q; k0 += 16) {
    f32x4 fa[2], fb[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = k0 + 4 * g + r, sc = s < cnt ? s : cnt - 1;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int d = 16 * (wave + 4 * x) + j;
        const float kv = a.kh[(row0 + sc) * HD + (long)h * D + (d < D ? d : D - 1)];
        fa[x][r] = s < cnt ? kv : 0.f;
      }
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const int p = p0 + 16 * y + j;
        const float vv = a.v[(row0 + sc) * a.ld + (long)h * Dv + (p < Dv ? p : Dv - 1)];
        fb[y][r] = s < cnt ? vv : 0.f;
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[x][y] = gla_mma(fa[x], fb[y], acc[x][y]);
  }
  float* dst = a.sc + ((long)(a.first(b) + blockIdx.y) * a.H + h) * D * Dv;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (wave + 4 * x) + 4 * g + r, p = p0 + 16 * y + j;
        if (d < D && p < Dv) dst[(long)d * Dv + p] = acc[x][y][r];
      }
}

// thread per state element of a (sequence, head), chunks in order (eight sums in flight); sc[c] becomes the START state of chunk c
__global__ __launch_bounds__(256) void gla_chunk_pass_kernel(float* __restrict__ state, GlaChunk a) {
  const int b = blockIdx.z, h = blockIdx.y;
  const long e = (long)blockIdx.x * 256 + threadIdx.x, NP = (long)a.D * a.Dv;
  if (e >= NP) return;
  const int nch = (a.seq_len[b] + GC_Q - 1) / GC_Q, d = (int)(e / a.Dv);
  if (nch == 0) return;
  float* sp = state + ((long)a.seq_slot[b] * a.H + h) * NP + e;
  float S = a.seq_pos0[b] == 0 ? 0.f : *sp;
  const long base = a.first(b), step = (long)a.H * NP;
  float* x = a.sc + (base * a.H + h) * NP + e;
  const float* ac = a.ac + (base * a.H + h) * a.D + d;
  for (int c0 = 0; c0 < nch; c0 += 8) {
    float add[8], dec[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = c0 + i < nch ? c0 + i : nch - 1;
      add[i] = x[c * step];
      dec[i] = ac[(long)c * a.H * a.D];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (c0 + i < nch) {
        x[(c0 + i) * step] = S;
        S = dec[i] * S + add[i];
      }
    }
  }
  *sp = S;
}

// grid (64-column slices, chunks, sequences x heads): wave w the read-outs of tokens 16 w .., four column tiles
__global__ __launch_bounds__(256) void gla_chunk_out_kernel(float* __restrict__ o, GlaChunk a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int LP = 68;
  const int b = blockIdx.z / a.H, h = blockIdx.z % a.H, t0 = blockIdx.y * GC_Q, len = a.seq_len[b];
  if (t0 >= len) return;
  const int cnt = len - t0 < GC_Q ? len - t0 : GC_Q, D = a.D, Dv = a.Dv, HD = a.H * D;
  const long row0 = (long)a.seq_row0[b] + t0;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4, p0 = blockIdx.x * 64;
  float* vs = sm;                          // [64][LP]
  float* ss = vs + GC_Q * LP;              // [D][LP]: the chunk's start state
  const float* s0 = a.sc + ((long)(a.first(b) + blockIdx.y) * a.H + h) * D * Dv;
  bool odd = false;                        // a value that is not finite
  for (int x = tid; x < (GC_Q + D) * 16; x += 256) {
    const int row = x >> 4, p = (x & 15) * 4, pc = p0 + p < Dv ? p0 + p : Dv - 4;
    const int t = row < GC_Q ? (row < cnt ? row : cnt - 1) : 0;
    const float* src = row < GC_Q ? a.v + (row0 + t) * a.ld + (long)h * Dv + pc : s0 + (long)(row - GC_Q) * Dv + pc;
    const f32x4 v = *reinterpret_cast<const f32x4*>(src);
    *reinterpret_cast<f32x4*>(sm + row * LP + p) = v;
    const f32x4 z = v - v;                 // zero, or NaN
    odd = odd || (row < GC_Q && !(z[0] + z[1] + z[2] + z[3] == 0.f));
  }
  const int t = 16 * wave + j, tc = t < cnt ? t : cnt - 1;
  f32x4 fm[4], fq[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) fm[i] = i <= wave ? *reinterpret_cast<const f32x4*>(a.m + ((row0 + tc) * a.H + h) * 64 + 16 * i + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 8; ++i) fq[i] = 16 * i < D ? *reinterpret_cast<const f32x4*>(a.qt + (row0 + tc) * HD + (long)h * D + 16 * i + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
  odd = __syncthreads_or(odd);
  f32x4 acc[4];
#pragma unroll
  for (int y = 0; y < 4; ++y) acc[y] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto cols = [&](const float* m, int k0, int y) {          // column 16 y + j, rows k0 + 4 g ..
    f32x4 f;
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = m[(k0 + 4 * g + r) * LP + 16 * y + j];
    return f;
  };
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (16 * i < D) {
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[y] = gla_mma(fq[i], cols(ss, 16 * i, y), acc[y]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i < wave || (i == wave && !odd)) {
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[y] = gla_mma(fm[i], cols(vs, 16 * i, y), acc[y]);
    }
  }
  if (odd) {                               // the wave's own block: no product with a later token's value
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tt = 16 * wave + 4 * g + r;
      const float* mr = a.m + ((row0 + (tt < cnt ? tt : cnt - 1)) * a.H + h) * 64;
      for (int u = 16 * wave; u <= tt; ++u)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[y][r] += mr[u] * vs[u * LP + 16 * y + j];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int tt = 16 * wave + 4 * g + r;
    if (tt >= cnt) continue;
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int p = p0 + 16 * y + j;
      if (p < Dv) o[(row0 + tt) * ((long)a.H * Dv) + (long)h * Dv + p] = acc[y][r] * a.qscale;
    }
  }
}

// floats of scratch for a step of T rows in B stretches; 0: the shape is not covered
extern "C" long umb_gla_scan_chunked_floats(int T, int B, int H, int D, int Dv) {
  if (T < 1 || B < 1 || H < 1 || D < 16 || D > 128 || D % 16 || Dv < 16 || Dv % 16) return 0;
  const long chunks = T / GC_Q + B;                          // whole chunks, and at most one started per stretch
  return (long)T * H * (2L * D + 64) + chunks * H * ((long)D * Dv + D);
}

extern "C" int umb_gla_scan_chunked(float* o, float* state, const float* proj, int ld, const float* log_alpha, const int* seq_slot,
                                    const int* seq_row0, const int* seq_pos0, const int* seq_len, int T, int B, int max_len, int H, int D, int Dv,
                                    float qscale, float* scratch, long scratch_floats, hipStream_t st) {
  const long need = umb_gla_scan_chunked_floats(T, B, H, D, Dv);
  if (need == 0 || need > scratch_floats || !o || !state || !proj || !log_alpha || !scratch || !seq_slot || !seq_row0 || !seq_pos0 || !seq_len ||
      max_len < 1 || max_len > T || (long)B * H > 65535 || ld < 2 * H * D + H * Dv || ld % 4 || ((uintptr_t)proj | (uintptr_t)scratch) % 16)
    return UMB_EINVAL;
  const int chunks = (max_len + GC_Q - 1) / GC_Q, HD = H * D;
  if (chunks > 65535) return UMB_EINVAL;
  const long nc = T / GC_Q + B;
  float* qt = scratch;
  float* kh = qt + (long)T * HD;
  float* m = kh + (long)T * HD;
  float* sc = m + (long)T * H * 64;
  float* ac = sc + nc * H * D * Dv;
  const GlaChunk a{proj, proj + HD, proj + 2L * HD, log_alpha, ld, H, D, Dv, seq_slot, seq_row0, seq_pos0, seq_len, qt, kh, m, sc, ac, qscale};
  const size_t lds1 = (2 * 5 * 128 + 4 * (size_t)GC_Q * (D + 4)) * sizeof(float), lds4 = (size_t)(GC_Q + D) * 68 * sizeof(float);
  if (ensure_dynamic_lds<gla_chunk_prep_kernel>(lds1) != UMB_OK || ensure_dynamic_lds<gla_chunk_out_kernel>(lds4) != UMB_OK) return UMB_EHIP;
  hipLaunchKernelGGL(gla_chunk_prep_kernel, dim3(chunks, H, B), dim3(1024), lds1, st, a);
  hipLaunchKernelGGL(gla_chunk_state_kernel, dim3((Dv + 63) / 64, chunks, B * H), dim3(256), 0, st, a);
  hipLaunchKernelGGL(gla_chunk_pass_kernel, dim3((unsigned)(((long)D * Dv + 255) / 256), H, B), dim3(256), 0, st, state, a);
  hipLaunchKernelGGL(gla_chunk_out_kernel, dim3((Dv + 63) / 64, chunks, B * H), dim3(256), lds4, st, o, a);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
