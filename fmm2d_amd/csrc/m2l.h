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
// workgroup 16 NW consecutive ones.  Per orbit and group of HB classes the
// wavefront loads its columns' source rows with consecutive lanes on
// consecutive coefficients (one group ahead, into registers), forms the z_c of
// each coefficient in the lane that holds its four sources, and keeps them in
// LDS, from where every lane reads its B operand; the operator's fragments of
// one class (v_mfma_*_16x16x4 A layout) are copied to LDS for the whole
// workgroup, two buffers deep and loaded two classes ahead.  The products of
// class a accumulate in their own tiles, so coefficients are padded to 8 RTC
// per class.
//
// What bounded the simpler forms (lfmm2d N = 1e7, 1.9e6 targets of 19
// coefficients): one operator per slot read through L1 by every wavefront,
// 50 GB of operators, 6.2 ms; orbits with each lane gathering its own
// components, 32 cache lines a load, 4.2 ms.  This form 3.8 ms: 40% of the
// cycles in MFMA, 52% with the LDS active; LDS latency between the chunks'
// barriers with two wavefronts per SIMD is what is left.
//
// All levels with the same tile shape go in one launch (the coarse levels of a
// Helmholtz tree are a few workgroups of serial latency each).  Neighbouring
// workgroups take the four child positions of the same parents, whose sources
// are mostly the same boxes, on one XCD.
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

// One level of a launch: child position q's targets are tlist[s0[q] .. s0[q] +
// n); P coefficients; boxes from box0 on, expansions from off on (complex
// values); operators from aoff on; first workgroup (of one child position) blk0.
struct M2LLev {
  int s0[4], n, P, box0, blk0;
  int64_t off, aoff;
};
constexpr int kM2LMaxLev = 52;
struct M2LTab {
  int nlev, nblk;  // workgroups per child position
  M2LLev lev[kM2LMaxLev];
};

template <typename T> struct M2LPair {
  T re, im;
};

template <typename T, int RTC, int KSC, int HB, int NW, int SGN, int LOGT>
__global__ __launch_bounds__(64 * NW) void k_m2l(int nd, int per_xcd, M2LTab tab,
                                                 const int* __restrict__ tlist,
                                                 const int* __restrict__ s2, M2LSlots orb,
                                                 const T* __restrict__ Aall,
                                                 const int* __restrict__ ilevel,
                                                 const int2* __restrict__ band,
                                                 const double* __restrict__ logr,
                                                 const cplx* __restrict__ srcall, cplx* dstall) {
  typedef typename Mfma<T>::acc_t acc_t;
  typedef M2LPair<T> pair_t;
  typedef M2LPair<double> dpair;
  constexpr int NT = 64 * NW;
  constexpr int CH = KSC * 4 * RTC * 64;  // values of one (orbit, b) chunk
  constexpr int NA = (CH + NT - 1) / NT;
  constexpr int CS = 2 * KSC;             // coefficients of a class, padded
  constexpr int JH = HB * CS;             // coefficients of a group
  constexpr int NIT = (16 * JH + 63) / 64;
  constexpr int NG = 4 / HB;              // groups of an orbit
  constexpr int ZS = JH + 1;              // z of a column, odd: reads without bank conflicts
  __shared__ T abuf[2][CH];
  __shared__ pair_t zbuf[NW][4][16][ZS];
  __shared__ int64_t offs[NW][2][16][4];
  __shared__ signed char slots[kM2LOrbits][4];
  const int64_t lblk = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (lblk >= 4 * (int64_t)tab.nblk) return;
  const int q = (int)(lblk & 3), pb = (int)(lblk >> 2);
  int li = 0;
  while (li + 1 < tab.nlev && pb >= tab.lev[li + 1].blk0) ++li;
  const int P = tab.lev[li].P, box0 = tab.lev[li].box0;
  const T* __restrict__ A = Aall + tab.lev[li].aoff;
  const dpair* __restrict__ src = reinterpret_cast<const dpair*>(srcall) + tab.lev[li].off;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, kr = lane >> 4, cl = lane & 15;
  if (tid < 4 * kM2LOrbits) (&slots[0][0])[tid] = (&orb.slot[q][0][0])[tid];
  const int64_t col = (int64_t)(pb - tab.lev[li].blk0) * (16 * NW) + wv * 16 + cl;
  const int64_t tpos = col / nd;
  const int d = (int)(col - tpos * nd);
  const int tb = tpos < tab.lev[li].n ? tlist[tab.lev[li].s0[q] + tpos] : -1;
  const int comp = kr & 1, jp = kr >> 1;
  acc_t acc[4][RTC];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < RTC; ++r) acc[a][r] = acc_t{0, 0, 0, 0};
  // FP32: z is formed in FP64 and rounded once, and the sums are folded into
  // FP64 ones after every second class of an orbit (hfmm2d N = 1e5, zk 30, eps
  // 1e-6: error against direct sums 1.1e-7, the kernel 0.39 ms; a fold an orbit
  // 1.5e-7, a little more than the one-source operators before it, and 0.29 ms; a
  // fold a class 1.0e-7, 0.42 ms; one chain over all orbits 3e-7)
  constexpr bool FOLD = sizeof(T) == 4;
  d4v sum[FOLD ? 4 : 1][FOLD ? RTC : 1];
#pragma unroll
  for (int a = 0; a < (FOLD ? 4 : 1); ++a)
#pragma unroll
    for (int r = 0; r < (FOLD ? RTC : 1); ++r) sum[a][r] = d4v{0, 0, 0, 0};
  double m0 = 0;
  __syncthreads();
  // The source of the orbit's kr-th rotation, as the offset of its expansion (-1:
  // none).  Loads are issued without branches, absent ones to a zero: a branch
  // around each load made the wavefront wait for its address first.
  int nextc = 0;
  auto load_c = [&](int o) {
    const int sl = o < kM2LOrbits ? slots[o][kr] : -1;
    nextc = s2[tb >= 0 && sl >= 0 ? (int64_t)kSlots * tb + sl : 0];
  };
  auto put_offs = [&](int o) {
    const int sl = o < kM2LOrbits ? slots[o][kr] : -1;
    offs[wv][o & 1][cl][kr] =
        tb >= 0 && sl >= 0 && nextc >= 0 ? ((int64_t)(nextc - box0) * nd + d) * P : -1;
  };
  // task `it` of a lane: coefficient jl of column tc of the wavefront's group
  dpair x[NIT][4];
  auto load_x = [&](int ob, int g) {
    int64_t of[NIT][4];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int t = min(it * 64 + lane, 16 * JH - 1), tc = t / JH;
#pragma unroll
      for (int k = 0; k < 4; ++k) of[it][k] = offs[wv][ob][tc][k];
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int t = min(it * 64 + lane, 16 * JH - 1), jl = t % JH;
      const int j = g * HB + (jl & (HB - 1)) + 4 * (jl / HB);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const dpair* p = of[it][k] >= 0 && j < P ? src + (of[it][k] + j)
                                                 : reinterpret_cast<const dpair*>(tr_zero);
        x[it][k] = *p;
      }
    }
  };
  auto store_z = [&]() {
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int t = it * 64 + lane, tc = t / JH, jl = t - tc * JH;
      const int row = (jl & (HB - 1)) * CS + jl / HB;
      if (16 * JH % 64 == 0 || t < 16 * JH) {
        const dpair s02{x[it][0].re + x[it][2].re, x[it][0].im + x[it][2].im};
        const dpair d02{x[it][0].re - x[it][2].re, x[it][0].im - x[it][2].im};
        const dpair s13{x[it][1].re + x[it][3].re, x[it][1].im + x[it][3].im};
        const dpair d13{x[it][1].re - x[it][3].re, x[it][1].im - x[it][3].im};
        zbuf[wv][0][tc][row] = pair_t{(T)(s02.re + s13.re), (T)(s02.im + s13.im)};
        zbuf[wv][1][tc][row] = pair_t{(T)(d02.re + d13.im), (T)(d02.im - d13.re)};  // - i d13
        zbuf[wv][2][tc][row] = pair_t{(T)(s02.re - s13.re), (T)(s02.im - s13.im)};
        zbuf[wv][3][tc][row] = pair_t{(T)(d02.re - d13.im), (T)(d02.im + d13.re)};
      }
    }
  };
  T ar[2][NA];
  auto load_a = [&](int chunk, T (&r)[NA]) {
    const T* p = A + (int64_t)chunk * CH + tid;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (CH % NT == 0 || NT * i + tid < CH) r[i] = p[NT * i];
  };
  auto store_a = [&](int buf, const T (&r)[NA]) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (CH % NT == 0 || NT * i + tid < CH) abuf[buf][NT * i + tid] = r[i];
  };
  constexpr int NCH = 4 * kM2LOrbits;
  load_a(0, ar[0]);
  load_a(1, ar[1]);
  load_c(0);
  put_offs(0);
  load_c(1);
  wave_lds_fence();
  load_x(0, 0);
  store_a(0, ar[0]);
  store_z();
  __syncthreads();
#pragma unroll 1
  for (int o = 0; o < kM2LOrbits; ++o) {
    const int ob = o & 1;
    put_offs(o + 1);
    wave_lds_fence();
    load_c(o + 2);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
      for (int u = 0; u < HB; ++u) {
        constexpr int one = 1;
        const int b = g * HB + u, cur = b & one, chunk = 4 * o + b;
        if (chunk + 2 < NCH) load_a(chunk + 2, ar[cur]);
        // the next group's rows (past the last orbit: none), after
        // the operator's loads: loads return in order, and the rows come from
        // farther away
        if (u == 0) {
          if (g + 1 < NG) load_x(ob, g + 1);
          else load_x(ob ^ 1, 0);
        }
#pragma unroll
        for (int ks = 0; ks < KSC; ++ks) {
          T z[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const pair_t* zp = &zbuf[wv][c][cl][u * CS + 2 * ks + jp];
            z[c] = reinterpret_cast<const T*>(zp)[comp];
          }
          if (LOGT && b == 0 && ks == 0) m0 += (double)z[0];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int a = (c - SGN * b) & 3;
#pragma unroll
            for (int r = 0; r < RTC; ++r)
              acc[a][r] = Mfma<T>::step(abuf[cur][((ks * 4 + c) * RTC + r) * 64 + lane], z[c],
                                        acc[a][r]);
          }
        }
        if (FOLD && (b & 1)) {
#pragma unroll
          for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int r = 0; r < RTC; ++r) {
#pragma unroll
              for (int i = 0; i < 4; ++i) sum[FOLD ? a : 0][FOLD ? r : 0][i] += (double)acc[a][r][i];
              acc[a][r] = acc_t{0, 0, 0, 0};
            }
        }
        if (chunk + 1 < NCH) store_a(cur ^ 1, ar[cur ^ 1]);
        __syncthreads();
      }
      store_z();
      wave_lds_fence();
    }
  }
  if (tb < 0) return;
  const int lev = ilevel[tb];
  const int2 bd = band ? band[lev] : int2{0, 2 * P};
  double* L = reinterpret_cast<double*>(dstall + tab.lev[li].off +
                                        ((int64_t)(tb - box0) * nd + d) * P);
  // the level-dependent part log(boxsize) M_0 of L_0: lanes 0..15 hold the
  // sources' sum of Re M_0, lanes 16..31 of Im M_0.  It is added by the lane that
  // adds the row's sum (FP64: the same lanes; FP32: rows 0 and 1 are both of
  // lanes 0..15), since nothing orders two lanes' updates of one value.
  const double lm = (LOGT && lane < 32) ? logr[lev] * m0 : 0.0;
  const double lmi = (LOGT && FOLD) ? __shfl(lm, cl + 16, 64) : lm;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < RTC; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * r + Mfma<T>::row(kr, i);
        const int e = 2 * (a + 4 * (row >> 1)) + (row & 1);
        if (e < 2 * P && e >= bd.x && e < bd.y) {
          double v = L[e];
          if constexpr (FOLD) v += sum[a][r][i];
          else v += acc[a][r][i];
          if (LOGT && a == 0 && row < 2) v += row == 0 ? lm : lmi;
          L[e] = v;
        }
      }
}

// The M2L of the given levels (blk0 is set here), one launch per tile shape.
// fp32: operators and z are float (sums of half an orbit FP32).  Every P <= kM2LMaxP;
// src and dst hold P values per (box, density) at the levels' off.
template <int SGN, int LOGT>
inline void launch_m2l(int nd, const std::vector<M2LLev>& levels, const int* tlist, const int* s2,
                       const void* A, const int* ilevel, const int2* band, const double* logr,
                       const cplx* src, cplx* dst, bool fp32, hipStream_t st) {
  const M2LSlots orb = m2l_orbit_slots();
  for (int ksc = 2; ksc <= 8; ++ksc) {
    const int nw = (!fp32 && ksc == 5) ? 8 : 4;
    M2LTab tab{};
    for (const M2LLev& v : levels) {
      if (m2l_ksc(v.P) != ksc || v.n <= 0) continue;
      if (tab.nlev == kM2LMaxLev) throw HipError{hipErrorInvalidValue, "m2l levels"};
      M2LLev& t = tab.lev[tab.nlev++];
      t = v;
      t.blk0 = tab.nblk;
      tab.nblk += (int)(((int64_t)v.n * nd + 16 * nw - 1) / (16 * nw));
    }
    if (tab.nlev == 0) continue;
    const int per_xcd = (int)((4 * (int64_t)tab.nblk + 7) / 8);
#define FMM2D_M2L(T, RTC, KSC, HB, NW)                                                         \
  hipLaunchKernelGGL((k_m2l<T, RTC, KSC, HB, NW, SGN, LOGT>), dim3((unsigned)(8 * per_xcd)),   \
                     dim3(64 * NW), 0, st, nd, per_xcd, tab, tlist, s2, orb,                   \
                     static_cast<const T*>(A), ilevel, band, logr, src, dst)
// Row tiles and k steps follow from P; HB, the classes that are transformed at a
// time, and the wavefronts:
// HB: with two classes transformed at a time a source row is loaded in two pieces
// and not four, but their z takes twice the LDS.  Two and three k steps: 2 (M2L
// of 1e6 points, 10 coefficients 0.37 ms, 0.42 with 1; 19 in FP32 0.32 and 0.38,
// of 1e7 in FP64 3.83 and 3.91).  Four k steps, where 2 leaves one workgroup a CU,
// have it too, though 1 is faster in FP64: 1e6 points with 29 coefficients 0.41 ms
// and 0.31 with 1, hfmm2d of 5e5 with 27 0.35 and 0.25.  From five on 1: 2
// takes 128 KB at five.
// Wavefronts: 8 share the operators where their z fits the LDS beside them and 4
// would leave one wavefront per SIMD, which is FP64 with five k steps alone (33 to
// 40 coefficients: 5e5 points with 39 0.50 ms, 0.63 with 4; 2e6 points with 17 to
// 201 4.1 and 5.1).  From six k steps on 8 do not fit the 163840 bytes of LDS
// (163880 at six) and FP64 stays at one wavefront per SIMD.
#define FMM2D_M2L_K(T, NW5)                   \
  switch (ksc) {                              \
    case 2: FMM2D_M2L(T, 1, 2, 2, 4); break;  \
    case 3: FMM2D_M2L(T, 1, 3, 2, 4); break;  \
    case 4: FMM2D_M2L(T, 1, 4, 2, 4); break;  \
    case 5: FMM2D_M2L(T, 2, 5, 1, NW5); break; \
    case 6: FMM2D_M2L(T, 2, 6, 1, 4); break;  \
    case 7: FMM2D_M2L(T, 2, 7, 1, 4); break;  \
    default: FMM2D_M2L(T, 2, 8, 1, 4); break; \
  }
    if (fp32) {
      FMM2D_M2L_K(float, 4)
    } else {
      FMM2D_M2L_K(double, 8)
    }
#undef FMM2D_M2L_K
#undef FMM2D_M2L
    hip_throw(hipGetLastError(), "m2l");
  }
}

}  // namespace fmm2d
