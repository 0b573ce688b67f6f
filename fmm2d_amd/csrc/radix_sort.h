// Stable LSD radix sort of 64-bit keys (optionally with 32-bit values) on the
// device: the point order of the tree build (common/pts_tree2d.f:1222-1246,
// pts_tree_sort, is a stable partition by the quadrant at every level; sorting
// the path keys is the same order).
//
// 8-bit digits, one launch per digit after one that counts the digits of every
// pass (k_rs_hist here, or the kernel that makes the keys, rs_count):
//   k_rs_pass: a workgroup takes the next tile of keys by ticket, ranks its
//   keys stably (the tile's waves, four or eight, take contiguous parts of it in
//   rounds of 64 consecutive keys: rank = keys of the digit in earlier waves +
//   earlier rounds + lower lanes), publishes its count of each digit, adds the
//   counts of the tiles before it by looking back over their published words (a
//   tile's own count, or the sum up to and including it: the decoupled look-back
//   of Merrill and Garland's single-pass scan, used for each digit as in Adinets
//   and Merrill's one-sweep radix sort), places its keys in
//   LDS in digit order and writes each digit's run with consecutive threads
//   on consecutive addresses.
// A tile waits only for tiles of earlier tickets, whose workgroups are already
// running and publish their counts before they wait, so every wait ends
// whatever else runs on the device.  Status words carry the pass in their tag, so
// they are cleared once per sort.
// Up to two arrays (sources and targets) are sorted by the same launches.
//
// Traffic per pass: keys and values read and written once.  Against a count,
// a scan and a scatter launch per digit (keys read twice): 15 launches to 6
// for a 40-bit sort of one array, 30 to 6 for two.
#pragma once
#include <algorithm>

#include "common.h"
#include "devbuf.h"
#include "scan.h"

namespace fmm2d {

constexpr int kRsMaxPass = 8;

// Lanes of the wave whose 8-bit digit equals this lane's (among `active`)
__device__ __forceinline__ unsigned long long rs_peers(unsigned d, unsigned long long active) {
  unsigned long long m = active;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const unsigned long long bal = __ballot((d >> b) & 1u);
    m &= ((d >> b) & 1u) ? bal : ~bal;
  }
  return m;
}

__device__ __forceinline__ unsigned long long rs_lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane ? (~0ull >> (64 - lane)) : 0ull;
}

// h[pass][digit] += the wave's keys (lanes with ok; call with the whole wave).
// In the top two passes, where neighbouring points share their digits, the
// highest lane of each group of equal digits adds the group's size (one LDS
// add and not up to 64 on one address); the lower digits differ from lane to
// lane, and finding the groups would cost more than the adds.
template <int NPASS>
__device__ __forceinline__ void rs_count(unsigned (*h)[256], unsigned long long key, bool ok,
                                         int npass) {
  const int lane = threadIdx.x & 63;
  const unsigned long long act = __ballot(ok);
#pragma unroll
  for (int p = 0; p < NPASS; ++p) {
    if (p >= npass) break;
    const unsigned d = (unsigned)(key >> (8 * p)) & 255u;
    if (p < npass - 2) {
      if (ok) atomicAdd(&h[p][d], 1u);
    } else {
      const unsigned long long m = rs_peers(d, act);
      if (ok && (m >> lane) == 1ull) atomicAdd(&h[p][d], (unsigned)__popcll(m));
    }
  }
}

// One array to sort: its keys and values of this pass, the digit counts
// [kRsMaxPass][256] of all its keys, and its tiles' status words [ntiles][256].
template <typename S> struct RsArray {
  const unsigned long long* kin;
  unsigned long long* kout;
  const int* vin;  // null in the first pass: the values are 0, 1, ...
  int* vout;
  int64_t n;
  int ntiles;
  const unsigned* hist;
  S* status;
};
template <typename S> struct RsPair {
  RsArray<S> a[2];
};

// status word: tag 2 pass + 1 (the tile's own count) or 2 pass + 2 (the count
// up to and including the tile) above kRsShift bits of count
template <typename S> struct RsWord;
template <> struct RsWord<unsigned> {
  static constexpr int shift = 27;
};
template <> struct RsWord<unsigned long long> {
  static constexpr int shift = 58;
};
constexpr int64_t kRsSmallMax = (int64_t(1) << 27) - 1;  // keys of 32-bit status words

template <typename S, int NT, int ITEMS, bool HAS_V>
__global__ __launch_bounds__(NT) void k_rs_pass(RsPair<S> pr, int pass, unsigned* ticket) {
  constexpr int TILE = NT * ITEMS;
  constexpr int NW = NT / 64;
  constexpr int WKEYS = TILE / NW;
  constexpr int SH = RsWord<S>::shift;
  constexpr S MASK = (S(1) << SH) - 1;
  __shared__ unsigned long long sk[TILE];
  __shared__ int sv[HAS_V ? TILE : 1];
  __shared__ unsigned wcnt[NW][256];
  __shared__ unsigned start[256];  // tile-local start of each digit's run
  __shared__ int64_t gbase[256];   // output position of the tile's first key of each digit
  __shared__ unsigned lds_scan[NW + 1];
  __shared__ int64_t lds_scan64[NW + 1];
  __shared__ int tk;
  if (threadIdx.x == 0) tk = (int)atomicAdd(ticket, 1u);
#pragma unroll
  for (int q = threadIdx.x; q < NW * 256; q += NT) (&wcnt[0][0])[q] = 0;
  __syncthreads();
  const int which = tk >= pr.a[0].ntiles ? 1 : 0;  // uniform
  const RsArray<S> A = pr.a[which];
  const int tile = tk - (which ? pr.a[0].ntiles : 0);
  const int shift = 8 * pass;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t tile0 = (int64_t)tile * TILE;
  const int64_t base = tile0 + (int64_t)w * WKEYS + lane;
  unsigned long long key[ITEMS];
  int val[ITEMS];
  unsigned long long peer[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t j = base + 64 * r;
    const bool ok = j < A.n;
    key[r] = ok ? A.kin[j] : 0ull;
    if (HAS_V) val[r] = ok ? (A.vin ? A.vin[j] : (int)j) : 0;
  }
  const bool isd = threadIdx.x < 256;
  const unsigned cnt_d = isd ? A.hist[256 * pass + threadIdx.x] : 0u;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool ok = base + 64 * r < A.n;
    const unsigned d = (unsigned)(key[r] >> shift) & 255u;
    peer[r] = rs_peers(d, __ballot(ok));
    if (ok && (peer[r] >> lane) == 1ull) wcnt[w][d] += (unsigned)__popcll(peer[r]);
  }
  __syncthreads();
  {
    // per digit (thread = digit): wave prefixes, tile-local start, the counts
    // of earlier tiles, output base
    const int d = threadIdx.x;
    unsigned s = 0;
    if (isd) {
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        const unsigned c = wcnt[q][d];
        wcnt[q][d] = s;
        s += c;
      }
    }
    S* mine = A.status + (int64_t)tile * 256 + (d & 255);
    const S own = S(2 * pass + 1) << SH, upto = S(2 * pass + 2) << SH;
    if (isd)
      __hip_atomic_store(mine, (tile == 0 ? upto : own) | S(s), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    unsigned tot;
    const unsigned st = block_exclusive_scan_w<NW>(s, lds_scan, &tot);
    int64_t tot64;
    const int64_t g = block_exclusive_scan_w<NW>((int64_t)cnt_d, lds_scan64, &tot64);
    if (isd) {
      start[d] = st;
#pragma unroll
      for (int q = 0; q < NW; ++q) wcnt[q][d] += st;  // running local positions
      // look back, kLook words in flight
      constexpr int kLook = 16;
      S before = 0;
      for (int t = tile - 1; t >= 0;) {
        S v[kLook];
#pragma unroll
        for (int u = 0; u < kLook; ++u)
          v[u] = t - u >= 0 ? __hip_atomic_load(A.status + (int64_t)(t - u) * 256 + d,
                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                            : upto;
        int used = 0;
        bool done = false;
#pragma unroll
        for (int u = 0; u < kLook; ++u) {
          const S tag = v[u] & ~MASK;
          if (used == u && !done && (tag == own || tag == upto)) {
            before += v[u] & MASK;
            ++used;
            done = tag == upto;
          }
        }
        if (done) break;
        t -= used;
      }
      if (tile > 0)
        __hip_atomic_store(mine, upto | (before + S(s)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      gbase[d] = g + (int64_t)before;
    }
  }
  __syncthreads();
  // stable ranks, keys placed in LDS in digit order
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool ok = base + 64 * r < A.n;
    const unsigned d = (unsigned)(key[r] >> shift) & 255u;
    unsigned pos = 0;
    if (ok) pos = wcnt[w][d] + (unsigned)__popcll(peer[r] & rs_lanemask_lt());
    __builtin_amdgcn_wave_barrier();  // every peer has read the running position
    if (ok && (peer[r] >> lane) == 1ull) wcnt[w][d] += (unsigned)__popcll(peer[r]);
    __builtin_amdgcn_wave_barrier();
    if (ok) {
      sk[pos] = key[r];
      if (HAS_V) sv[pos] = val[r];
    }
  }
  __syncthreads();
  const int cnt = (int)min((int64_t)TILE, A.n - tile0);
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int p = r * NT + threadIdx.x;
    if (p >= cnt) break;
    const unsigned long long k = sk[p];
    const unsigned d = (unsigned)(k >> shift) & 255u;
    const int64_t dst = gbase[d] + (p - (int)start[d]);
    A.kout[dst] = k;
    if (HAS_V) A.vout[dst] = sv[p];
  }
}

// digit counts of every pass into hist[pass][digit] (cleared by the caller)
constexpr int kRsCountThreads = 1024;
// workgroups that count digits: each adds its counts with one global atomic
// per digit and pass, which contend (2048 workgroups: 83 us for 2e6 keys)
inline unsigned rs_count_grid(int64_t n) {
  return (unsigned)std::min<int64_t>(512, std::max<int64_t>(1, ceil_div(n, kRsCountThreads)));
}
static __global__ __launch_bounds__(kRsCountThreads) void k_rs_hist(
    const unsigned long long* __restrict__ keys, int64_t n, int npass, unsigned* hist) {
  __shared__ unsigned h[kRsMaxPass][256];
  for (int q = threadIdx.x; q < kRsMaxPass * 256; q += kRsCountThreads) (&h[0][0])[q] = 0;
  __syncthreads();
  for (int64_t i0 = (int64_t)blockIdx.x * kRsCountThreads; i0 < n;
       i0 += (int64_t)gridDim.x * kRsCountThreads) {
    const int64_t i = i0 + threadIdx.x;
    rs_count<kRsMaxPass>(h, i < n ? keys[i] : 0ull, i < n, npass);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < npass * 256; q += kRsCountThreads)
    if ((&h[0][0])[q]) atomicAdd(&hist[q], (&h[0][0])[q]);
}

// Tiles of 512 and 1024 keys for small arrays (more workgroups, shorter chains
// inside one), 4096 for large ones, where the look-back over the tiles in
// flight counts.
struct RsTile {
  int nt, items;
};
inline RsTile rs_tile(int64_t n) {
  return n <= 16384 ? RsTile{256, 2} : n <= 262144 ? RsTile{256, 4} : RsTile{512, 8};
}

// The buffers of one sort of up to two arrays.  `clear` words must be zero
// before the digits are counted (hist) and the first pass runs.
struct RsPlan {
  int64_t n[2] = {0, 0};
  int npass = 0;
  RsTile shape{512, 8};
  int ntiles[2] = {0, 0};
  bool wide = false;     // 64-bit status words
  DBuf<unsigned> words;  // hist[2][npass][256], tickets[npass], status
  size_t status0 = 0;    // first status word
  unsigned* hist(int k) const { return words.p + (size_t)256 * npass * k; }
  unsigned* tickets() const { return words.p + (size_t)512 * npass; }

  void init(int64_t n0, int64_t n1, int bits, hipStream_t st) {
    n[0] = n0;
    n[1] = n1;
    npass = (std::max(bits, 1) + 7) / 8;
    const int64_t m = std::max(n0, n1);
    shape = rs_tile(m);
    wide = m > kRsSmallMax;
    const int64_t tile = (int64_t)shape.nt * shape.items;
    for (int k = 0; k < 2; ++k) ntiles[k] = (int)((n[k] + tile - 1) / tile);
    status0 = ((size_t)512 * npass + npass + 63) / 64 * 64;
    words.alloc(status0 + (size_t)256 * (ntiles[0] + ntiles[1]) * (wide ? 2 : 1), st);
  }

  template <typename S, int NT, int ITEMS, bool HAS_V>
  void launch(const RsPair<S>& pr, int p, hipStream_t st) const {
    hipLaunchKernelGGL((k_rs_pass<S, NT, ITEMS, HAS_V>), dim3(ntiles[0] + ntiles[1]), dim3(NT), 0,
                       st, pr, p, tickets() + p);
  }
  template <typename S, bool HAS_V>
  void passes(const unsigned long long* const* kin, unsigned long long* const* kout,
              const int* const* vin, int* const* vout, hipStream_t st) const {
    DBuf<unsigned long long> kt[2];
    DBuf<int> vt[2];
    if (npass > 1)
      for (int k = 0; k < 2; ++k) {
        kt[k].alloc(n[k], st);
        if (HAS_V) vt[k].alloc(n[k], st);
      }
    RsPair<S> pr{};
    for (int p = 0; p < npass; ++p) {
      // the last pass writes kout: odd passes from the end go to the scratch
      const bool to_out = ((npass - 1 - p) % 2) == 0;
      S* stat = reinterpret_cast<S*>(words.p + status0);
      for (int k = 0; k < 2; ++k) {
        RsArray<S>& a = pr.a[k];
        a.kin = p == 0 ? kin[k] : a.kout;
        a.vin = p == 0 ? (vin ? vin[k] : nullptr) : a.vout;
        a.kout = to_out ? kout[k] : kt[k].p;
        a.vout = HAS_V ? (to_out ? vout[k] : vt[k].p) : nullptr;
        a.n = n[k];
        a.ntiles = ntiles[k];
        a.hist = hist(k);
        a.status = stat + (size_t)256 * (k ? ntiles[0] : 0);
      }
      if constexpr (sizeof(S) == 8) {
        launch<S, 512, 8, HAS_V>(pr, p, st);
      } else {
        if (shape.items == 2) launch<S, 256, 2, HAS_V>(pr, p, st);
        else if (shape.items == 4) launch<S, 256, 4, HAS_V>(pr, p, st);
        else launch<S, 512, 8, HAS_V>(pr, p, st);
      }
      hip_throw(hipGetLastError(), "radix sort");
    }
  }
  // kin / vin are not modified; kout (and vout, unless null) receive the
  // result.  vin null: values 0, 1, ....  n = 0 arrays may have null pointers.
  void sort(const unsigned long long* const* kin, unsigned long long* const* kout,
            const int* const* vin, int* const* vout, hipStream_t st) const {
    if (ntiles[0] + ntiles[1] == 0 || npass == 0) return;
    if (wide) {
      if (vout) passes<unsigned long long, true>(kin, kout, vin, vout, st);
      else passes<unsigned long long, false>(kin, kout, vin, vout, st);
    } else {
      if (vout) passes<unsigned, true>(kin, kout, vin, vout, st);
      else passes<unsigned, false>(kin, kout, vin, vout, st);
    }
  }
};

// Stable sort of n keys by their low `bits` (<= 64) bits with values.
// vin null: values 0, 1, ...; vout null: keys alone.
inline void radix_sort(const unsigned long long* kin, unsigned long long* kout, const int* vin,
                       int* vout, int64_t n, int bits, hipStream_t st) {
  if (n <= 0) return;
  RsPlan P;
  P.init(n, 0, bits, st);
  P.words.zero();
  hipLaunchKernelGGL(k_rs_hist, dim3(rs_count_grid(n)), dim3(kRsCountThreads), 0, st, kin, n,
                     P.npass, P.hist(0));
  hip_throw(hipGetLastError(), "radix sort");
  const unsigned long long* ki[2] = {kin, nullptr};
  unsigned long long* ko[2] = {kout, nullptr};
  const int* vi[2] = {vin, nullptr};
  int* vo[2] = {vout, nullptr};
  P.sort(ki, ko, vin ? vi : nullptr, vout ? vo : nullptr, st);
}

}  // namespace fmm2d
