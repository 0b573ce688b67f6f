// Device-wide exclusive prefix sums (the role of common/cumsum.f:39 in the
// reference's tree build, and of the offset scans of the drivers).
//
// A thread holds kScanItems elements, kScanQ rounds of kScanV consecutive ones
// (all loads issued before the first is used, consecutive lanes on consecutive
// 16-byte pieces), and a workgroup scans its kScanQ x 256 thread sums with one
// wave64 shuffle scan.  The arrays of a tree build are a few thousand to a few
// million elements, so the cost is launches and memory latency, not bytes:
//   n <= kScanSingleMax   one workgroup, one launch (256 threads for a single
//                         tile, whose 4 waves' sums add faster than 16);
//   up to kScanLookMax    tile sums, then every workgroup adds the sums of the
//                         tiles before its own and scans its tile: two
//                         launches;
//   beyond                tile sums, their scan by one workgroup, the tiles:
//                         three launches (the re-added sums would grow with the
//                         square of the tiles).
// MI355X: 50k elements 63 -> 8 us and 32k elements 30 -> 8 us against one
// workgroup whose threads each walked a contiguous chunk (uncoalesced, the
// loads of a chunk in series); 1.25e6 elements (three launches before) 23 -> 16.
// Deterministic (fixed summation order), in place allowed (out == in).
#pragma once
#include "common.h"
#include "devbuf.h"

namespace fmm2d {

constexpr int kScanThreads = 256;
constexpr int kScanWaves = kScanThreads / 64;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanThreads * kScanItems;

// Exclusive scan of v over a workgroup of NW waves; *total = the sum.  lds
// holds NW + 1 values.  Ends with a barrier, so lds may be reused.
template <int NW, typename T>
__device__ __forceinline__ T block_exclusive_scan_w(T v, T* lds, T* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  T x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) lds[w] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    T s = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const T t = lds[i];
      lds[i] = s;
      s += t;
    }
    lds[NW] = s;
  }
  __syncthreads();
  const T ex = x - v + lds[w];
  *total = lds[NW];
  __syncthreads();
  return ex;
}

// the same over a workgroup of kScanThreads (256) threads
template <typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* lds, T* total) {
  return block_exclusive_scan_w<kScanWaves>(v, lds, total);
}

// kScanItems elements of thread `threadIdx.x` of a workgroup of NT threads from
// base on (0 beyond n), the sum of each round's kScanV in sum[]
constexpr int kScanV = 4, kScanQ = kScanItems / kScanV;

template <int NT, typename T>
__device__ __forceinline__ void scan_load(const T* in, int64_t base, int64_t n, T v[kScanQ][kScanV],
                                          T sum[kScanQ]) {
#pragma unroll
  for (int q = 0; q < kScanQ; ++q) {
    const int64_t j = base + ((int64_t)q * NT + threadIdx.x) * kScanV;
    if (j + kScanV <= n) {
#pragma unroll
      for (int e = 0; e < kScanV; ++e) v[q][e] = in[j + e];
    } else {
#pragma unroll
      for (int e = 0; e < kScanV; ++e) v[q][e] = j + e < n ? in[j + e] : T(0);
    }
  }
#pragma unroll
  for (int q = 0; q < kScanQ; ++q) {
    sum[q] = v[q][0];
#pragma unroll
    for (int e = 1; e < kScanV; ++e) sum[q] += v[q][e];
  }
}

// Scans the tile at base (NT x kScanItems elements) and writes it, starting
// from carry; returns the tile's total (on every thread).
template <int NT, typename T>
__device__ __forceinline__ T scan_tile(const T* in, T* out, int64_t base, int64_t n, T carry) {
  constexpr int NW = NT / 64;
  __shared__ T lds[kScanQ][NW];
  T v[kScanQ][kScanV], s[kScanQ], x[kScanQ];
  scan_load<NT>(in, base, n, v, s);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < kScanQ; ++q) x[q] = s[q];
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
    for (int q = 0; q < kScanQ; ++q) {
      const T y = __shfl_up(x[q], d, 64);
      if (lane >= d) x[q] += y;
    }
  }
  if (lane == 63) {
#pragma unroll
    for (int q = 0; q < kScanQ; ++q) lds[q][w] = x[q];
  }
  __syncthreads();
  // the waves before this one in round q, after the rounds before q
  T tot = 0;
#pragma unroll
  for (int q = 0; q < kScanQ; ++q) {
    if (base + (int64_t)q * NT * kScanV >= n) break;  // uniform
    T before = carry + tot;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const T t = lds[q][i];
      if (i < w) before += t;
      tot += t;
    }
    T run = before + x[q] - s[q];
    const int64_t j = base + ((int64_t)q * NT + threadIdx.x) * kScanV;
    T o[kScanV];
#pragma unroll
    for (int e = 0; e < kScanV; ++e) {
      o[e] = run;
      run += v[q][e];
    }
    if (j + kScanV <= n) {
#pragma unroll
      for (int e = 0; e < kScanV; ++e) out[j + e] = o[e];
    } else {
#pragma unroll
      for (int e = 0; e < kScanV; ++e)
        if (j + e < n) out[j + e] = o[e];
    }
  }
  return tot;
}

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const T* __restrict__ in,
                                                              int64_t n, T* part) {
  __shared__ T lds[kScanWaves + 1];
  T v[kScanQ][kScanV], q[kScanQ];
  scan_load<kScanThreads>(in, (int64_t)blockIdx.x * kScanTile, n, v, q);
  T s = q[0];
#pragma unroll
  for (int i = 1; i < kScanQ; ++i) s += q[i];
  T tot;
  block_exclusive_scan(s, lds, &tot);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// One workgroup: exclusive scan of the nblk tile sums in place.
template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_top(T* part, int64_t nblk) {
  __shared__ T lds[kScanWaves + 1];
  T carry = 0;
  for (int64_t b0 = 0; b0 < nblk; b0 += kScanThreads) {
    const int64_t j = b0 + threadIdx.x;
    const T v = j < nblk ? part[j] : T(0);
    T tot;
    const T ex = block_exclusive_scan(v, lds, &tot);
    if (j < nblk) part[j] = carry + ex;
    carry += tot;
  }
}

// The tiles.  LOOK: part holds the tile sums and the workgroup adds those
// before its own; else their exclusive scan.
template <typename T, bool LOOK>
__global__ __launch_bounds__(kScanThreads) void k_scan_down(const T* in, T* out, int64_t n,
                                                            const T* part, T* total) {
  __shared__ T lds[kScanWaves + 1];
  T carry = 0;
  if (LOOK) {
    T s = 0;
    for (int64_t j = threadIdx.x; j < blockIdx.x; j += kScanThreads) s += part[j];
    block_exclusive_scan(s, lds, &carry);
  } else {
    carry = part[blockIdx.x];
  }
  const T tot = scan_tile<kScanThreads>(in, out, (int64_t)blockIdx.x * kScanTile, n, carry);
  if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = carry + tot;
}

constexpr int kScan1Threads = 1024;
constexpr int64_t kScanSingleMax = kScan1Threads * kScanItems;
constexpr int64_t kScanLookMax = 2048 * kScanTile;

template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_scan_single(const T* in, T* out, int64_t n, T* total) {
  const T tot = scan_tile<NT>(in, out, 0, n, T(0));
  if (threadIdx.x == 0 && total) *total = tot;
}

// out[i] = in[0] + ... + in[i-1] for i < n; *total (device, may be null) =
// the sum of all n.  Stream-ordered, no host synchronisation.
template <typename T>
void exclusive_scan(const T* in, T* out, int64_t n, T* total, hipStream_t st) {
  if (n <= 0) {
    if (total) hip_throw(hipMemsetAsync(total, 0, sizeof(T), st), "hipMemsetAsync");
    return;
  }
  if (n <= kScanSingleMax) {
    if (n <= kScanTile)
      hipLaunchKernelGGL((k_scan_single<T, kScanThreads>), dim3(1), dim3(kScanThreads), 0, st, in, out,
                         n, total);
    else
      hipLaunchKernelGGL((k_scan_single<T, kScan1Threads>), dim3(1), dim3(kScan1Threads), 0, st, in,
                         out, n, total);
    hip_throw(hipGetLastError(), "scan");
    return;
  }
  const int64_t nblk = ceil_div(n, (int64_t)kScanTile);
  DBuf<T> part(nblk, st);
  hipLaunchKernelGGL(k_scan_reduce<T>, dim3(nblk), dim3(kScanThreads), 0, st, in, n, part.p);
  if (n <= kScanLookMax) {
    hipLaunchKernelGGL((k_scan_down<T, true>), dim3(nblk), dim3(kScanThreads), 0, st, in, out, n,
                       (const T*)part.p, total);
  } else {
    hipLaunchKernelGGL(k_scan_top<T>, dim3(1), dim3(kScanThreads), 0, st, part.p, nblk);
    hipLaunchKernelGGL((k_scan_down<T, false>), dim3(nblk), dim3(kScanThreads), 0, st, in, out, n,
                       (const T*)part.p, total);
  }
  hip_throw(hipGetLastError(), "scan");
}

}  // namespace fmm2d
