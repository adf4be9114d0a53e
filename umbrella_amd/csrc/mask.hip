// A boolean attention mask [T][C] (columns are cache slots) as the tree-attention kernels read it: the columns every row attends in front
// become a prefix length, what follows becomes bit rows.
//
// Replaces the mask handling of the reference's Llama.inference (umbrella/models/llama.py:117-134, where flashinfer takes the boolean
// mask itself).  Latency alone: a few KB to a few hundred KB.  As array expressions this was some twenty launches and four host round
// trips in front of a forward; now two launches and one round trip.  A whole call, before -> now: one row behind 900 cached tokens 980
// -> 837 us, 257 rows of a 70B AWQ model 3030 -> 2809 us.
#include "common.h"
#include "../../include/umbrella_hip.h"

// out[2 b], out[2 b + 1] of 64-column block b: its first column that some row does not attend (C: none), one past its last column
// that some row attends (0: none); out[2 blocks] = max(slots).  Workgroup: lane = column, wave = every 16th row.
__global__ __launch_bounds__(1024) void mask_scan_kernel(int* __restrict__ out, const unsigned char* __restrict__ mask, long ld, int T, int C,
                                                         const void* __restrict__ slots, int slots64) {
  __shared__ unsigned long long all_s[16], any_s[16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c0 = blockIdx.x * 64, c = min(c0 + lane, C - 1);
  bool all = true, any = false;
#pragma unroll 8
  for (int r = wave; r < T; r += 16) {
    const bool v = mask[(long)r * ld + c] != 0;
    all = all && v;
    any = any || v;
  }
  const unsigned long long a = __ballot(all || c0 + lane >= C), o = __ballot(any && c0 + lane < C);
  if (lane == 0) { all_s[wave] = a; any_s[wave] = o; }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long A = ~0ull, O = 0ull;
#pragma unroll
    for (int w = 0; w < 16; ++w) { A &= all_s[w]; O |= any_s[w]; }
    out[2 * blockIdx.x] = A == ~0ull ? C : c0 + __ffsll(~A) - 1;
    out[2 * blockIdx.x + 1] = O ? c0 + 64 - __clzll(O) : 0;
  }
  if (blockIdx.x == 0 && wave == 1) {
    int m = 0;
    for (int r = lane; r < T; r += 64) m = max(m, slots64 ? (int)static_cast<const long long*>(slots)[r] : static_cast<const int*>(slots)[r]);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) m = max(m, __shfl_xor(m, s, 64));
    if (lane == 0) out[2 * gridDim.x] = m;
  }
}

// bits[t][w] = columns prefix + 64 w .. of row t; idx = {ids [T], positions [T], slots [T], prefix} in 32 bits.  One wave per bit word.
__global__ __launch_bounds__(256) void mask_pack_kernel(unsigned long long* __restrict__ bits, int W, int* __restrict__ idx,
                                                        const unsigned char* __restrict__ mask, long ld, int T, int C, int prefix,
                                                        const void* __restrict__ ids, int ids64, const void* __restrict__ pos, int pos64,
                                                        const void* __restrict__ slots, int slots64) {
  const int lane = threadIdx.x & 63;
  const long n = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n < (long)T * W) {
    const int t = (int)(n / W), c = prefix + (int)(n % W) * 64 + lane;
    const unsigned long long b = __ballot(c < C && mask[(long)t * ld + min(c, C - 1)] != 0);
    if (lane == 0) bits[n] = b;
  }
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < 3L * T) {
    const int which = (int)(i / T), t = (int)(i % T);
    const void* src = which == 0 ? ids : which == 1 ? pos : slots;
    const int wide = which == 0 ? ids64 : which == 1 ? pos64 : slots64;
    idx[i] = wide ? (int)static_cast<const long long*>(src)[t] : static_cast<const int*>(src)[t];
  } else if (i == 3L * T) {
    idx[i] = prefix;
  }
}

extern "C" int umb_mask_scan(int* out, const void* mask, long ld, int T, int C, const void* slots, int slots64, hipStream_t st) {
  if (T < 1 || C < 1 || ld < C || !out || !mask || !slots) return UMB_EINVAL;
  hipLaunchKernelGGL(mask_scan_kernel, dim3((C + 63) / 64), dim3(1024), 0, st, out, (const unsigned char*)mask, ld, T, C, slots, slots64);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}

extern "C" int umb_mask_pack(void* bits, int W, int* idx, const void* mask, long ld, int T, int C, int prefix, const void* ids, int ids64,
                             const void* pos, int pos64, const void* slots, int slots64, hipStream_t st) {
  if (T < 1 || C < 1 || ld < C || W < 1 || prefix < 0 || !bits || !idx || !mask || !ids || !pos || !slots) return UMB_EINVAL;
  const long words = ((long)T * W + 3) / 4, conv = (3L * T + 1 + 255) / 256;
  hipLaunchKernelGGL(mask_pack_kernel, dim3((unsigned)(words > conv ? words : conv)), dim3(256), 0, st, (unsigned long long*)bits, W, idx,
                     (const unsigned char*)mask, ld, T, C, prefix, ids, ids64, pos, pos64, slots, slots64);
  UMB_LAUNCH_CHECK();
  return UMB_OK;
}
