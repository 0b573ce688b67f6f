// Multipole-to-local translations of long expansions (more than 64
// coefficients, beyond m2l.h) on MFMA, shared by the Laplace/Cauchy and
// Helmholtz drivers.
//
// A translation is y = T x with T a complex Pout x Pin operator and x, y box
// expansions.  In real form T becomes a 2Pout x 2Pin matrix over interleaved
// (re, im) coefficients; operators are pre-swizzled into the A-operand layout
// of v_mfma_f64_16x16x4f64 (lane l holds row l%16, column l/16 of a 16x4
// block; the result tile holds row l/16 + 4 i, column l%16 in element i).
//
// Slot s of target t reads source slots[t * nslots + s] (-1: empty).
// Work is split into groups: group g owns targets tlist[seg0[g]..seg1[g])
// and tiles [tile0[g], tile0[g+1]) of 16 columns; within a group every target has the same
// slot -> operator map (opbase[g] + slot_op[cls[g]*nslots + s]), so the A
// operand is uniform across a wavefront, whose 16 columns are (target,
// density) pairs: dst[t] += sum_s T_s src[slot(t,s)].  Box b's expansion for density d
// starts at ((b - box0) nd + d) P of its buffer (box0 = first box of the
// buffer's level, 0 for a buffer holding all levels).  With a band table,
// band[level] = [lo, hi) are the interleaved coefficient rows that level uses
// (the rest stay zero); without one every row is used.  With LOGT the Laplace
// M2L term log(boxsize) M_0 is added to L_0.
//
// The k loop is bound by the latency of its loads, operator fragments from L2
// and one coefficient a lane: the fragments of all row tiles of a step and the
// coefficient are in flight together, and the number of row tiles is a constant
// of each copy of the loop, so that nothing in it is in a branch.  With the row
// tiles under a test, each MFMA waited for its own load (and, where the test was
// of a vector register, moved its accumulators to vector registers and back):
// M2L of hfmm2d at eps 1e-12, 5e5 points (67 to 75 coefficients) 5.95 -> 3.2
// ms, 3e5 points on a curve (67 to 185) 11.3 -> 5.7.
#pragma once
#include <type_traits>
#include <vector>

#include "common.h"
#include "devbuf.h"

namespace fmm2d {

typedef double d4v __attribute__((ext_vector_type(4)));

// Group table of one launch, passed by value: group g owns targets
// tlist[seg0[g]..seg1[g]) and tiles [tile0[g], tile0[g+1]).
constexpr int kTrMaxGroups = 8;
// Groups of one launch.  Wave tiles: the first ilv tiles of every group go
// round-robin over the groups (tile t of group g is wave t * ng + g), the
// rest group after group from ng * ilv on (group g's from rem0[g]); ilv = 0
// is group after group throughout.  Interleaving the M2L classes (the four
// child positions) puts siblings, whose list-2 sources are mostly the same
// boxes, into neighbouring waves of one workgroup.
// row tiles accumulated per pass over the k steps
constexpr int kTrRows = 4;

struct TrTable {
  int ng, ilv;
  int tile0[kTrMaxGroups + 1];
  int rem0[kTrMaxGroups + 1];
  int seg0[kTrMaxGroups], seg1[kTrMaxGroups];
  int opbase[kTrMaxGroups], cls[kTrMaxGroups];
};

typedef float f4v __attribute__((ext_vector_type(4)));

// One 16x16x4 MFMA step in the element type T (double: v_mfma_f64_16x16x4f64,
// float: v_mfma_f32_16x16x4f32), and the output row of accumulator element i
// for lane group kr: the two instructions lay their 16x16 results out
// differently (f64: row kr + 4 i, f32: row 4 kr + i).
template <typename T> struct Mfma;
template <> struct Mfma<double> {
  typedef d4v acc_t;
  static __device__ __forceinline__ acc_t step(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int kr, int i) { return kr + 4 * i; }
};
template <> struct Mfma<float> {
  typedef f4v acc_t;
  static __device__ __forceinline__ acc_t step(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int kr, int i) { return 4 * kr + i; }
};

// orders a wavefront's LDS writes before its later LDS reads and vice versa
// (the wavefront's LDS accesses complete in order; this keeps the compiler
// from moving them across)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

static __device__ double tr_zero[2];  // what an absent coefficient is loaded from

// T is the arithmetic type of the operator (Afrag) and the source
// expansions (src, 2 Pin values of T per box and density); the results are
// added to the FP64 destination expansions.
template <typename T, int LOGT>
__global__ __launch_bounds__(256) void k_translate(
    int nd, int P, int nslots, int64_t nwaves, int per_xcd, TrTable tab, const int* tlist,
    const int* slots, const int* slot_op, const T* Afrag, int64_t afs, int box0,
    const int* ilevel, const int2* band, const double* logr, const T* src, cplx* dst, int ssplit,
    int ksplit, double* part, int64_t* dstoff) {
  typedef typename Mfma<T>::acc_t acc_t;
  constexpr int RT = kTrRows;
  // Workgroups are dispatched round-robin over the 8 XCDs; block b works on
  // logical block (b % 8) * per_xcd + b / 8 so that each XCD walks a
  // contiguous range of targets, whose neighbouring source boxes then stay
  // in that XCD's L2.
  const int64_t lblk = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  // (the wavefront's number as a scalar: with the row tile's bound a vector
  // condition every MFMA stood in a branch of its own, its accumulators moved to
  // vector registers and back around it)
  const int64_t wv0 = lblk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wv0 >= nwaves) return;
  const int lane = threadIdx.x & 63;
  // Split launches (few targets, long operators): wavefront wv0 also takes
  // one of ssplit groups of slots and one of ksplit ranges of k steps.  It
  // writes the partial sums of group sk to part[sk][column][row] (all 16 RTT
  // rows, 0 outside the band) and the target's offset in dst to
  // dstoff[column], for k_tr_split_sum to add in group order.
  const int nsk = ssplit * ksplit;
  const int sk = (int)(wv0 % nsk);
  const int64_t wv = wv0 / nsk;
  const bool split = nsk > 1;
  // The chunks of RT row tiles go to separate wavefronts: wavefront wv works
  // on tile wv / nrc, chunk wv % nrc (the rows are disjoint outputs).
  const int RTT = (2 * P + 15) / 16, KS = (2 * P + 3) / 4;
  const int nrc = (RTT + RT - 1) / RT;
  const int64_t wave = wv / nrc;
  const int rc = (int)(wv - wave * nrc) * RT;
  int g = 0;
  int64_t tl;  // tile within group g
  if (wave < (int64_t)tab.ilv * tab.ng) {
    g = (int)(wave % tab.ng);
    tl = wave / tab.ng;
  } else {
    const int64_t w2 = wave - (int64_t)tab.ilv * tab.ng;
    while (g + 1 < tab.ng && w2 >= tab.rem0[g + 1]) ++g;
    tl = tab.ilv + (w2 - tab.rem0[g]);
  }
  const int q = tab.cls[g];
  const int64_t col = tl * 16 + (lane & 15);
  const int64_t tpos = tab.seg0[g] + col / nd;
  const int d = (int)(col % nd);
  // a target list entry may be -1 (no target at that position)
  const int tb = tpos < tab.seg1[g] ? tlist[tpos] : -1;
  const bool valid = tb >= 0;
  const int kr = lane >> 4;
  if (__ballot(valid) == 0) {
    // no target in the tile
    if (split && sk == 0 && rc == 0 && kr == 0)
      dstoff[(int64_t)(tab.tile0[g] + tl) * 16 + (lane & 15)] = -1;
    return;
  }
  const int2 full = int2{0, 2 * P};
  const int ob = tab.opbase[g];
  const int sg = sk / ksplit, kg = sk - sg * ksplit;
  const int s_lo = (int)((int64_t)nslots * sg / ssplit);
  const int s_hi = (int)((int64_t)nslots * (sg + 1) / ssplit);
  const int k_lo = (int)((int64_t)KS * kg / ksplit);
  const int k_hi = (int)((int64_t)KS * (kg + 1) / ksplit);
  acc_t acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = acc_t{0, 0, 0, 0};
  T m0 = 0;
  auto products = [&](auto NRC) {
    constexpr int NR = decltype(NRC)::value;  // row tiles of this chunk
    for (int s = s_lo; s < s_hi; ++s) {
      const int c = valid ? slots[(int64_t)tb * nslots + s] : -1;
      const T* A = Afrag + (int64_t)(ob + slot_op[q * nslots + s]) * afs + lane;
      const T* M = src + (c >= 0 ? ((int64_t)(c - box0) * nd + d) * 2 * P : 0);
      int klo = 0, khi = 0;
      if (c >= 0) {
        const int2 bd = band ? band[ilevel[c]] : full;
        klo = bd.x;
        khi = bd.y;
      }
#pragma unroll 2
      for (int ks = k_lo; ks < k_hi; ++ks) {
        const int k = 4 * ks + kr;
        T av[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) av[r] = A[((int64_t)(rc + r) * KS + ks) * 64];
        // (absent coefficients are loaded from a zero: no load in a branch)
        const T b = *((k >= klo && k < khi) ? M + k : reinterpret_cast<const T*>(tr_zero));
        if (LOGT && rc == 0 && ks == 0 && lane < 32) m0 += b;
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[r] = Mfma<T>::step(av[r], b, acc[r]);
      }
    }
  };
  switch (min(RT, RTT - rc)) {
    case 1: products(std::integral_constant<int, 1>{}); break;
    case 2: products(std::integral_constant<int, 2>{}); break;
    case 3: products(std::integral_constant<int, 3>{}); break;
    default: products(std::integral_constant<int, RT>{}); break;
  }
  if (split) {
    const int64_t ncols = (int64_t)tab.tile0[tab.ng] * 16;
    const int64_t colg = (int64_t)(tab.tile0[g] + tl) * 16 + (lane & 15);
    double* Pp = part + ((int64_t)sk * ncols + colg) * (16 * RTT);
    if (sk == 0 && rc == 0 && kr == 0)
      dstoff[colg] = valid ? ((int64_t)(tb - box0) * nd + d) * 2 * P : -1;
    const int2 bd = valid ? (band ? band[ilevel[tb]] : full) : int2{0, 0};
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * (rc + r) + Mfma<T>::row(kr, i);
        if (rc + r < RTT) Pp[row] = (row >= bd.x && row < bd.y) ? (double)acc[r][i] : 0.0;
      }
  } else if (valid) {
    const int2 bd = band ? band[ilevel[tb]] : full;
    double* L = reinterpret_cast<double*>(dst + ((int64_t)(tb - box0) * nd + d) * P);
    // level-dependent part of L_0: lanes 0..15 hold Re M_0 (row 0), lanes
    // 16..31 Im M_0 (row 1) of their column
    if (LOGT && rc == 0 && lane < 32) L[kr] += logr[ilevel[tb]] * (double)m0;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * (rc + r) + Mfma<T>::row(kr, i);
        if (rc + r < RTT && row >= bd.x && row < bd.y) L[row] += (double)acc[r][i];
      }
  }
}

// Real interleaved form of square complex operators ops[o][j][n] (input j,
// output n), swizzled as Afrag[o][row tile][k step][lane].
template <typename T = double>
inline std::vector<T> swizzle_ops(int P, const std::vector<cplx>& ops, int nops) {
  const int K2 = 2 * P, RTT = (K2 + 15) / 16, KS = (K2 + 3) / 4;
  std::vector<T> out((size_t)nops * RTT * KS * 64, T(0));
  for (int o = 0; o < nops; ++o)
    for (int r = 0; r < RTT; ++r)
      for (int ks = 0; ks < KS; ++ks)
        for (int l = 0; l < 64; ++l) {
          const int row = 16 * r + (l & 15), col = 4 * ks + (l >> 4);
          double v = 0.0;
          if (row < K2 && col < K2) {
            const cplx t = ops[((size_t)o * P + col / 2) * P + row / 2];
            const int a = row & 1, b = col & 1;
            v = (a == b) ? t.re : (a == 0 ? -t.im : t.im);
          }
          out[(((size_t)o * RTT + r) * KS + ks) * 64 + l] = (T)v;
        }
  return out;
}

// values per swizzled operator of P x P complex entries
inline int64_t afrag_stride(int P) {
  return (int64_t)((2 * P + 15) / 16) * ((2 * P + 3) / 4) * 64;
}

struct TrGroup {
  int seg0, seg1;  // targets tlist[seg0..seg1)
  int opbase, cls;
};

// dst[dstoff[c] + row] += sum over the nsk split groups, in group order, of
// part[k][c][row] (rows 0 .. rows-1 of the ncols columns; dstoff -1: none)
static __global__ void k_tr_split_sum(int64_t n, int64_t ncols, int rstride, int rows, int nsk,
                               const double* __restrict__ part, const int64_t* __restrict__ dstoff,
                               double* dst) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t c = t / rows;
  const int row = (int)(t - c * rows);
  const int64_t o = dstoff[c];
  if (o < 0) return;
  double s = 0.0;
  for (int k = 0; k < nsk; ++k) s += part[((int64_t)k * ncols + c) * rstride + row];
  dst[o + row] += s;
}

// Launch translate passes over the given groups (at most kTrMaxGroups per
// launch; launches are stream-ordered, so groups must not depend on each other).
// fp32: operators (Afrag) and sources are float, accumulation FP32 on
// v_mfma_f32_16x16x4f32; otherwise FP64.  src, dst: the expansions of the
// boxes from box0 on, P coefficients each.
// Launches with fewer wavefronts than this split their slots and their k steps
// over more wavefronts, whose partial sums are added in a fixed order (no
// atomics: the results do not depend on scheduling): small problems and coarse
// levels would otherwise run a few dozen wavefronts through 27 slots each.
constexpr int64_t kTrSplitWaves = 4096;

template <typename T, int LOGT>
void launch_translate(int nd, int P, const void* src, cplx* dst, int box0, int nslots,
                      const std::vector<TrGroup>& groups, const int* tlist, const int* slots,
                      const int* slot_op, const void* Afrag, const int* ilevel, const int2* band,
                      const double* logr, hipStream_t st) {
  const int64_t afs = afrag_stride(P);
  const int RTT = (2 * P + 15) / 16, KS = (2 * P + 3) / 4;
  size_t gi = 0;
  while (gi < groups.size()) {
    TrTable tab{};
    int tiles = 0;
    for (; gi < groups.size() && tab.ng < kTrMaxGroups; ++gi) {
      const TrGroup& g = groups[gi];
      if (g.seg1 <= g.seg0) continue;
      tab.tile0[tab.ng] = tiles;
      tab.seg0[tab.ng] = g.seg0;
      tab.seg1[tab.ng] = g.seg1;
      tab.opbase[tab.ng] = g.opbase;
      tab.cls[tab.ng] = g.cls;
      ++tab.ng;
      tiles += (int)(((int64_t)(g.seg1 - g.seg0) * nd + 15) / 16);
    }
    if (tab.ng == 0) continue;
    tab.tile0[tab.ng] = tiles;
    tab.ilv = tiles;
    for (int g = 0; g < tab.ng; ++g) tab.ilv = std::min(tab.ilv, tab.tile0[g + 1] - tab.tile0[g]);
    tab.rem0[0] = 0;
    for (int g = 0; g < tab.ng; ++g)
      tab.rem0[g + 1] = tab.rem0[g] + (tab.tile0[g + 1] - tab.tile0[g]) - tab.ilv;
    const int64_t nw0 = (int64_t)tiles * ((RTT + kTrRows - 1) / kTrRows);
    int ssplit = 1, ksplit = 1;
    if (!LOGT && nw0 < kTrSplitWaves) {
      ssplit = (int)std::min<int64_t>(nslots, (kTrSplitWaves + nw0 - 1) / nw0);
      ksplit = (int)std::max<int64_t>(
          1, std::min<int64_t>(KS / 16, (kTrSplitWaves + nw0 * ssplit - 1) / (nw0 * ssplit)));
    }
    const int nsk = ssplit * ksplit;
    const int64_t nw = nw0 * nsk;
    const int per_xcd = (int)(((nw + 3) / 4 + 7) / 8);
    // partial sums per (split group, column)
    const int64_t ncols = (int64_t)tiles * 16;
    DBuf<double> part(nsk > 1 ? (size_t)nsk * ncols * 16 * RTT : 0, st);
    DBuf<int64_t> dstoff(nsk > 1 ? (size_t)ncols : 0, st);
    hipLaunchKernelGGL((k_translate<T, LOGT>), dim3((unsigned)(8 * per_xcd)), dim3(256), 0, st,
                       nd, P, nslots, nw, per_xcd, tab, tlist, slots, slot_op,
                       static_cast<const T*>(Afrag), afs, box0, ilevel, band, logr,
                       static_cast<const T*>(src), dst, ssplit, ksplit, part.p, dstoff.p);
    if (nsk > 1)
      launch1d(k_tr_split_sum, ncols * 2 * P, st, ncols, 16 * RTT, 2 * P, nsk,
               (const double*)part.p, (const int64_t*)dstoff.p, reinterpret_cast<double*>(dst));
    hip_throw(hipGetLastError(), "translate");
  }
}

}  // namespace fmm2d
