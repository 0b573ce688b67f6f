// Multipole-to-local translations of one level (Helmholtz) or the whole tree
// (Laplace) for expansions of up to 64 coefficients, shared by both drivers
// (l2dmploc, laprouts2d.f:1130-1244; h2dmploc, helmrouts2d.f:1221-1382).
//
// Four sources at the offsets u, iu, -u, -iu of a target have one operator up
// to phases:  T(i^k u)[n][j] = i^{-k (n + j)} T(u)[n][j]  (Laplace; Helmholtz
// i^{-k (n - j)}), so with the coefficients split by residue mod 4 (n = a,
// j = b)
//   out_a = sum_b T_ab z_c,b,   z_c = sum_k i^{-k c} x_k,   c = a + b (a - b),
// and one operator serves four sources after a 4-point DFT of their
// coefficients (eight additions for four values).  The 27 offsets of a child
// position are 10 such orbits (four full ones, five of two sources, one
// single), so a target takes 10 operators' worth of matrix work and not 27.
//
// A wavefront owns 16 (target, density) columns of one child position, a
// workgroup 64 consecutive ones; per (orbit, b) chunk the operator's fragments
// (v_mfma_*_16x16x4 A layout) are copied to LDS once for the four wavefronts,
// two buffers deep, and every lane loads its component of the four sources'
// coefficients one chunk ahead, into registers.  The products of class a
// accumulate in their own tiles, so coefficients are padded to 8 RTC per
// class.  (Per-wavefront operators read through L1 were the bound before: 15
// KB a slot and wavefront, 50 GB over the 1.9e6 targets of lfmm2d N = 1e7.)
//
// Neighbouring workgroups take the four child positions of the same parents,
// whose sources are mostly the same boxes, on one XCD.
#pragma once
#include <vector>

#include "common.h"
#include "devbuf.h"
#include "translate.h"
#include "tree.h"

namespace fmm2d {

constexpr int kM2LOrbits = 10;
constexpr int kM2LMaxP = 64;
// one offset of each orbit; the others are its rotations by 90 degrees
constexpr int kM2LBase[kM2LOrbits][2] = {{2, 0}, {2, 1}, {1, 2}, {2, 2}, {3, 0},
                                         {3, 1}, {1, 3}, {3, 2}, {2, 3}, {3, 3}};

// slot[q][o][k]: the offset slot of orbit o's k-th rotation for child position
// q, -1 where q has none
struct M2LSlots {
  signed char slot[4][kM2LOrbits][4];
};
inline M2LSlots m2l_orbit_slots() {
  M2LSlots s;
  for (int q = 0; q < 4; ++q)
    for (int o = 0; o < kM2LOrbits; ++o) {
      int dx = kM2LBase[o][0], dy = kM2LBase[o][1];
      for (int k = 0; k < 4; ++k) {
        s.slot[q][o][k] = (signed char)m2l_slot(q, dx, dy);
        const int t = dx;
        dx = -dy;
        dy = t;
      }
    }
  return s;
}

// k steps (of 4 interleaved coefficients) per class and row tiles per class
inline int m2l_ksc(int P) { return std::max(2, ((P + 3) / 4 + 1) / 2); }
inline int m2l_rtc(int P) { return ((P + 3) / 4 + 7) / 8; }
// values of one operator: [b][k step][c][row tile][lane]
inline int64_t m2l_stride(int P) { return (int64_t)4 * m2l_ksc(P) * 4 * m2l_rtc(P) * 64; }

// Coefficients (output n, input j; real row, column parts) of fragment value e
// of an operator; n or j may be P or more (padding).
struct M2LEntry {
  int n, j, rpart, cpart;
};
FMM2D_HD M2LEntry m2l_entry(int e, int ksc, int rtc, int sgn) {
  const int lane = e & 63;
  int t = e >> 6;
  const int r = t % rtc;
  t /= rtc;
  const int c = t & 3;
  t >>= 2;
  const int ks = t % ksc, b = t / ksc;
  const int a = (c - sgn * b) & 3;
  const int row = 16 * r + (lane & 15), col = 4 * ks + (lane >> 4);
  return M2LEntry{a + 4 * (row >> 1), b + 4 * (col >> 1), row & 1, col & 1};
}

// Operators T[o] (complex P x P, entry [j * P + n]) in fragment layout
template <typename T>
inline std::vector<T> m2l_swizzle(int P, const std::vector<std::vector<cplx>>& ops, int sgn) {
  const int ksc = m2l_ksc(P), rtc = m2l_rtc(P);
  const int64_t st = m2l_stride(P);
  std::vector<T> out((size_t)(st * (int64_t)ops.size()), T(0));
  for (size_t o = 0; o < ops.size(); ++o)
    for (int64_t e = 0; e < st; ++e) {
      const M2LEntry m = m2l_entry((int)e, ksc, rtc, sgn);
      if (m.n >= P || m.j >= P) continue;
      const cplx t = ops[o][(size_t)m.j * P + m.n];
      out[(size_t)(o * st + e)] =
          (T)(m.rpart == m.cpart ? t.re : (m.rpart == 0 ? -t.im : t.im));
    }
  return out;
}

// Targets of one launch: child position q's are tlist[s0[q] .. s0[q] + n)
struct M2LSeg {
  int s0[4], n;
};

template <typename T, int RTC, int KSC, int SGN, int LOGT>
__global__ __launch_bounds__(256) void k_m2l(int nd, int P, int nblk, int per_xcd, M2LSeg seg,
                                             const int* __restrict__ tlist,
                                             const int* __restrict__ s2, M2LSlots orb,
                                             const T* __restrict__ A, int sbox0, int dbox0,
                                             const int* __restrict__ ilevel,
                                             const int2* __restrict__ band,
                                             const double* __restrict__ logr,
                                             const T* __restrict__ src, cplx* dst) {
  typedef typename Mfma<T>::acc_t acc_t;
  constexpr int CH = KSC * 4 * RTC * 64;  // values of one (orbit, b) chunk
  constexpr int NA = CH / 256;
  __shared__ T abuf[2][CH];
  __shared__ signed char slots[kM2LOrbits][4];
  const int64_t lblk = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (lblk >= 4 * (int64_t)nblk) return;
  const int q = (int)(lblk & 3);
  const int tid = threadIdx.x, lane = tid & 63, kr = lane >> 4;
  if (tid < 4 * kM2LOrbits) (&slots[0][0])[tid] = (&orb.slot[q][0][0])[tid];
  const int64_t col = (lblk >> 2) * 64 + (tid >> 6) * 16 + (lane & 15);
  const int64_t tpos = col / nd;
  const int d = (int)(col - tpos * nd);
  const int tb = tpos < seg.n ? tlist[seg.s0[q] + tpos] : -1;
  const int comp = kr & 1, jp = kr >> 1;
  const T sg = comp ? T(-1) : T(1);
  acc_t acc[4][RTC];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < RTC; ++r) acc[a][r] = acc_t{0, 0, 0, 0};
  // FP32: every orbit's sums are folded into FP64 ones (a long FP32 chain over
  // the orbits doubled the error of hfmm2d, zk 30, eps 1e-6)
  constexpr bool FOLD = sizeof(T) == 4;
  d4v sum[FOLD ? 4 : 1][FOLD ? RTC : 1];
#pragma unroll
  for (int a = 0; a < (FOLD ? 4 : 1); ++a)
#pragma unroll
    for (int r = 0; r < (FOLD ? RTC : 1); ++r) sum[a][r] = d4v{0, 0, 0, 0};
  double m0 = 0;
  __syncthreads();
  // the source of the orbit's kr-th rotation
  auto my_source = [&](int o) {
    const int sl = slots[o][kr];
    return (tb >= 0 && sl >= 0) ? s2[(int64_t)kSlots * tb + sl] : -1;
  };
  const T* px[4];
  auto set_sources = [&](int myc) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int c = __shfl(myc, (lane & 15) + 16 * k, 64);
      px[k] = c >= 0 ? src + ((int64_t)(c - sbox0) * nd + d) * 2 * P + comp : nullptr;
    }
  };
  T v[2][KSC][4];
  auto load_x = [&](int b, T (&w)[KSC][4]) {
#pragma unroll
    for (int ks = 0; ks < KSC; ++ks) {
      const int j = b + 4 * (2 * ks + jp);
#pragma unroll
      for (int k = 0; k < 4; ++k) w[ks][k] = (px[k] && j < P) ? px[k][2 * j] : T(0);
    }
  };
  T ar[NA];
  auto load_a = [&](int chunk) {
    const T* p = A + (int64_t)chunk * CH + tid;
#pragma unroll
    for (int i = 0; i < NA; ++i) ar[i] = p[256 * i];
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i) abuf[buf][256 * i + tid] = ar[i];
  };
  set_sources(my_source(0));
  load_x(0, v[0]);
  load_a(0);
  store_a(0);
  __syncthreads();
#pragma unroll 1
  for (int o = 0; o < kM2LOrbits; ++o) {
    const int nextc = o + 1 < kM2LOrbits ? my_source(o + 1) : -1;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      constexpr int one = 1;
      const int cur = b & one;
      const bool more = b < 3 || o + 1 < kM2LOrbits;
      if (more) {
        load_a(4 * o + b + 1);
        if (b == 3) set_sources(nextc);
        load_x((b + 1) & 3, v[cur ^ 1]);
      }
#pragma unroll
      for (int ks = 0; ks < KSC; ++ks) {
        const T s02 = v[cur][ks][0] + v[cur][ks][2], d02 = v[cur][ks][0] - v[cur][ks][2];
        const T s13 = v[cur][ks][1] + v[cur][ks][3], d13 = v[cur][ks][1] - v[cur][ks][3];
        const T o13 = sg * __shfl_xor(d13, 16, 64);  // the other component, for -+i d13
        const T z[4] = {s02 + s13, d02 + o13, s02 - s13, d02 - o13};
        if (LOGT && b == 0 && ks == 0) m0 += (double)z[0];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int a = (c - SGN * b) & 3;
#pragma unroll
          for (int r = 0; r < RTC; ++r)
            acc[a][r] =
                Mfma<T>::step(abuf[cur][((ks * 4 + c) * RTC + r) * 64 + lane], z[c], acc[a][r]);
        }
      }
      if (more) store_a(cur ^ 1);
      __syncthreads();
    }
    if constexpr (FOLD) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int r = 0; r < RTC; ++r) {
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[a][r][i] += (double)acc[a][r][i];
          acc[a][r] = acc_t{0, 0, 0, 0};
        }
    }
  }
  if (tb < 0) return;
  const int lev = ilevel[tb];
  const int2 bd = band ? band[lev] : int2{0, 2 * P};
  double* L = reinterpret_cast<double*>(dst + ((int64_t)(tb - dbox0) * nd + d) * P);
  // the level-dependent part log(boxsize) M_0 of L_0: lanes 0..15 hold the
  // sources' sum of Re M_0, lanes 16..31 of Im M_0
  const double lm = (LOGT && lane < 32) ? logr[lev] * m0 : 0.0;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < RTC; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * r + Mfma<T>::row(kr, i);
        const int e = 2 * (a + 4 * (row >> 1)) + (row & 1);
        if (e < 2 * P && e >= bd.x && e < bd.y) {
          if constexpr (FOLD) L[e] += sum[a][r][i];
          else L[e] += acc[a][r][i];
        }
      }
  if (LOGT && lane < 32) L[kr] += lm;
}

// One M2L launch.  fp32: operators and sources are float (an orbit's sums FP32).  P <= kM2LMaxP.
template <int SGN, int LOGT>
inline void launch_m2l(int nd, int P, const M2LSeg& seg, const int* tlist, const int* s2,
                       const void* A, int sbox0, int dbox0, const int* ilevel, const int2* band,
                       const double* logr, const void* src, cplx* dst, bool fp32,
                       hipStream_t st) {
  if (seg.n <= 0) return;
  const M2LSlots orb = m2l_orbit_slots();
  const int64_t nblk = ((int64_t)seg.n * nd + 63) / 64;
  const int per_xcd = (int)((4 * nblk + 7) / 8);
#define FMM2D_M2L(T, RTC, KSC)                                                                  \
  hipLaunchKernelGGL((k_m2l<T, RTC, KSC, SGN, LOGT>), dim3((unsigned)(8 * per_xcd)), dim3(256), \
                     0, st, nd, P, (int)nblk, per_xcd, seg, tlist, s2, orb,                     \
                     static_cast<const T*>(A), sbox0, dbox0, ilevel, band, logr,                \
                     static_cast<const T*>(src), dst)
#define FMM2D_M2L_K(T)                \
  switch (m2l_ksc(P)) {               \
    case 2: FMM2D_M2L(T, 1, 2); break; \
    case 3: FMM2D_M2L(T, 1, 3); break; \
    case 4: FMM2D_M2L(T, 1, 4); break; \
    case 5: FMM2D_M2L(T, 2, 5); break; \
    case 6: FMM2D_M2L(T, 2, 6); break; \
    case 7: FMM2D_M2L(T, 2, 7); break; \
    default: FMM2D_M2L(T, 2, 8); break; \
  }
  if (fp32) {
    FMM2D_M2L_K(float)
  } else {
    FMM2D_M2L_K(double)
  }
#undef FMM2D_M2L_K
#undef FMM2D_M2L
  hip_throw(hipGetLastError(), "m2l");
}

}  // namespace fmm2d
