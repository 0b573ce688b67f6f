// Multipole-to-multipole and local-to-local translations between a box and its
// four children (l2dmpmp, l2dlocloc, laprouts2d.f:912-1124; h2dmpmp,
// h2dlocloc, helmrouts2d.f:967-1215), one launch per level, shared by the
// Laplace/Cauchy and Helmholtz drivers.
//
// The children's offsets are u, iu, -u, -iu with u = (1, 1): their operators
// are one operator T up to phases, T_k[n][m] = i^{s k e} T[n][m] with e = n - m
// (orders) and s = -1, but s = +1 for the Laplace M2M.  With c = e mod 4,
//   M2M: parent[n] = sum_m T[n][m] X_c[m],    X_c[m] = sum_k i^{s k c} child_k[m]
//   L2L: child_k[n] = sum_c i^{s k c} Y_c[n], Y_c[n] = sum_{m in c} T[n][m] parent[m]
// so a 4-point DFT on one side leaves one product with T per parent, a quarter
// of the arithmetic, which is then small beside the memory traffic even on the
// vector units: nothing is padded to matrix tiles, and every shape runs the
// same code.
//
// A thread owns one row n of NP (parent, density) columns; T is stored so that
// for the step (t, c) all rows read consecutive values (m = 4 t + the residue
// that belongs to n and c), and their operands X_c[m] are four consecutive
// values in LDS.  Long expansions run through LDS in chunks.  Few columns: the
// steps of a row are also split over MG threads, added in a fixed order.
//
// What bounded the MFMA form (16 columns of one wavefront against four
// operators, and a second kernel adding the partial sums of small levels):
// latency.  A level took 8-10 us for 19 coefficients and 17-22 us for 61, of
// which the memory traffic of the small ones is nothing and that of the
// largest a third.  This form: lfmm2d N = 1e7 (13 levels, 19 coefficients,
// 1.8e6 boxes) 1.52 -> 0.68 ms for both directions, hfmm2d at 2e6 points (16
// levels, up to 201 coefficients) 2.64 -> 0.55 ms; a level of 470 parents 5 us; the
// largest level moves its 320 MB at 3.7 TB/s.
#pragma once
#include <algorithm>

#include "common.h"
#include "devbuf.h"

namespace fmm2d {

constexpr int kShiftT = 256;         // threads of a workgroup
constexpr int kShiftLds = 40 << 10;  // bytes of staged values

// Coefficients of one (box, density): stride values apart, the first n used
// (the rest are zero and stay so); box b's start at ((b - box0) nd + d) stride.
struct ShiftSide {
  cplx* p;
  int box0, stride, n;
};

struct ShiftShape {
  int rows, tiles;  // rows of a tile, tiles
  int mg, pg;       // threads per row, column groups of a workgroup
  int mc;           // staged coefficients per chunk (a multiple of 4)
};

// complex values of an operator with nin columns and nout rows; entry e is
// T[n][m] (m >= nin: zero), see shift_entry
__host__ __device__ inline int64_t shift_stride(int nin, int nout) {
  return (int64_t)((nin + 3) / 4) * 4 * nout;
}

// row n, column m of value e; sh = (order of row 0) - (order of column 0)
__host__ __device__ __forceinline__ void shift_entry(int64_t e, int nout, int sh, int* n, int* m) {
  *n = (int)(e % nout);
  const int tc = (int)(e / nout);
  *m = 4 * (tc >> 2) + ((*n + sh - (tc & 3)) & 3);
}

// x i^k
__device__ __forceinline__ cplx mul_i(cplx x, int k) {
  k &= 3;
  return k == 0 ? x : k == 1 ? cplx{-x.im, x.re} : k == 2 ? cplx{-x.re, -x.im} : cplx{x.im, -x.re};
}

// UP: M2M (src: children, dst: parents, assigned); else L2L (src: parents, dst:
// children, added to).  slots[4 i + q]: the child of parent i = parents[i] in
// position q (bit 0: right, bit 1: upper), or -1.
template <int UP, int SGN, int NP>
__global__ __launch_bounds__(kShiftT) void k_shift(int64_t ncols, int nd, ShiftShape s, int sh,
                                                   const int* __restrict__ parents,
                                                   const int4* __restrict__ slots, ShiftSide src,
                                                   ShiftSide dst, const cplx* __restrict__ A) {
  extern __shared__ cplx xs[];
  const int tid = threadIdx.x;
  const int nc = s.pg * NP;  // columns of the workgroup
  const int64_t col0 = (int64_t)blockIdx.x * nc;
  const int row = tid % s.rows, grp = tid / s.rows;
  const int mg = grp % s.mg, pg = grp / s.mg;
  const int n = blockIdx.y * s.rows + row;
  const bool on = pg < s.pg && n < dst.n;
  constexpr int NY = UP ? 1 : 4;
  cplx acc[NP][NY];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int y = 0; y < NY; ++y) acc[p][y] = cplx{0.0, 0.0};

  // L2L: the values that the sums go to, on their way while the sums form
  int64_t at[NP][4];
  cplx old[NP][UP ? 1 : 4];
  if (!UP) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int64_t col = col0 + pg * NP + p;
      const bool ok = on && mg == 0 && col < ncols;
      const int64_t i = ok ? col / nd : 0;
      const int d = ok ? (int)(col - i * nd) : 0;
      const int4 ch = slots[i];
      const int c4[4] = {ch.w, ch.z, ch.x, ch.y};  // k = 0..3
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        at[p][k] = ok && c4[k] >= 0 ? ((int64_t)(c4[k] - dst.box0) * nd + d) * dst.stride + n : -1;
        old[p][k] = dst.p[at[p][k] >= 0 ? at[p][k] : 0];
      }
    }
  }

  const int nt = (src.n + 3) / 4;  // steps t of a whole row
  for (int m0 = 0; m0 < 4 * nt; m0 += s.mc) {
    const int mc = min(s.mc, 4 * nt - m0);
    if (m0) __syncthreads();
    for (int e = tid; e < nc * mc; e += kShiftT) {
      const int j = e / mc, m = m0 + e - j * mc;
      const int64_t col = col0 + j;
      const bool ok = col < ncols && m < src.n;
      const int64_t i = ok ? col / nd : 0;
      const int d = ok ? (int)(col - i * nd) : 0;
      if (UP) {
        const int4 ch = slots[i];
        const int c4[4] = {ch.w, ch.z, ch.x, ch.y};
        cplx x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool has = ok && c4[k] >= 0;
          const cplx v =
              src.p[has ? ((int64_t)(c4[k] - src.box0) * nd + d) * src.stride + m : 0];
          x[k] = has ? v : cplx{0.0, 0.0};
        }
        const cplx a = x[0] + x[2], b = x[0] - x[2], f = x[1] + x[3], g = mul_i(x[1] - x[3], 1);
        cplx* o = xs + (int64_t)j * 4 * mc + (m - m0);
        o[0] = a + f;
        o[mc] = SGN > 0 ? b + g : b - g;
        o[2 * mc] = a - f;
        o[3 * mc] = SGN > 0 ? b - g : b + g;
      } else {
        const cplx v =
            src.p[ok ? ((int64_t)(parents[i] - src.box0) * nd + d) * src.stride + m : 0];
        xs[e] = ok ? v : cplx{0.0, 0.0};
      }
    }
    __syncthreads();
    if (on) {
      const int nts = mc / 4, per = (nts + s.mg - 1) / s.mg;
      const int t0 = mg * per, t1 = min(nts, t0 + per);
      const cplx* a = A + ((int64_t)(m0 / 4 + t0) * 4) * dst.stride + n;
      int res[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) res[c] = (n + sh - c) & 3;
#pragma unroll 2
      for (int t = t0; t < t1; ++t) {
        cplx av[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) av[c] = a[(int64_t)c * dst.stride];
        a += (int64_t)4 * dst.stride;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            const int j = pg * NP + p;
            const cplx x = UP ? xs[(j * 4 + c) * mc + 4 * t + res[c]] : xs[j * mc + 4 * t + res[c]];
            cplx& y = acc[p][UP ? 0 : c];
            y.re = fma(av[c].re, x.re, fma(-av[c].im, x.im, y.re));
            y.im = fma(av[c].re, x.im, fma(av[c].im, x.re, y.im));
          }
      }
    }
  }
  if (s.mg > 1) {  // sums over the MG threads of a row, in order (NP = 1)
    __syncthreads();
    if (on && mg > 0)
#pragma unroll
      for (int y = 0; y < NY; ++y)
        xs[((pg * (s.mg - 1) + mg - 1) * NY + y) * s.rows + row] = acc[0][y];
    __syncthreads();
    if (on && mg == 0)
      for (int g = 1; g < s.mg; ++g)
#pragma unroll
        for (int y = 0; y < NY; ++y)
          acc[0][y] = acc[0][y] + xs[((pg * (s.mg - 1) + g - 1) * NY + y) * s.rows + row];
  }
  if (!on || mg != 0) return;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    if (UP) {
      const int64_t col = col0 + pg * NP + p;
      if (col >= ncols) break;
      const int64_t i = col / nd;
      const int d = (int)(col - i * nd);
      dst.p[((int64_t)(parents[i] - dst.box0) * nd + d) * dst.stride + n] = acc[p][0];
    } else {
      const cplx y0 = acc[p][0], y1 = acc[p][NY > 1 ? 1 : 0], y2 = acc[p][NY > 1 ? 2 : 0],
                 y3 = acc[p][NY > 1 ? 3 : 0];
      const cplx a = y0 + y2, b = y0 - y2, f = y1 + y3, g = mul_i(y1 - y3, 1);
      const cplx out[4] = {a + f, SGN > 0 ? b + g : b - g, a - f, SGN > 0 ? b - g : b + g};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (at[p][k] >= 0) dst.p[at[p][k]] = old[p][UP ? 0 : k] + out[k];
    }
  }
}

// One level: np parents (parents, slots: their entries of the level), operator
// A of shift_stride(src.stride, dst.stride) values for the child in position 3,
// sh = (order of row 0) - (order of column 0).
//
// Large levels: two columns a thread, whole rows.  Below 512 workgroups of that
// form: one column a thread, tiles of at most 32 rows and the row's steps over
// up to nt/3 threads.  Measured, large form against small: L2L of 16 parents
// with 201 coefficients 99 / 15 us, of 470 parents with 19 7.4 / 6.6; equal at
// 500 workgroups (M2M 10.1 / 10.0, 10.5 / 14.5); M2M of 27000 parents with 41
// coefficients 44 / 68 us.
template <int UP, int SGN>
void launch_shift(int nd, int np, const int* parents, const int* slots, const ShiftSide& src,
                  const ShiftSide& dst, int sh, const cplx* A, hipStream_t st) {
  if (np <= 0 || src.n <= 0 || dst.n <= 0) return;
  const int64_t ncols = (int64_t)np * nd;
  const int nt = (src.n + 3) / 4;
  auto shape = [&](int maxrows) {
    ShiftShape s{};
    s.tiles = (dst.n + maxrows - 1) / maxrows;
    s.rows = (dst.n + s.tiles - 1) / s.tiles;
    s.mg = 1;
    s.pg = std::min(kShiftT / s.rows, 32);
    return s;
  };
  ShiftShape s = shape(64);
  int npar = 2;
  if ((ncols + 2 * s.pg - 1) / (2 * s.pg) * s.tiles < 512) {
    s = shape(32);
    npar = 1;
    s.mg = std::max(1, std::min(s.pg, nt / 3));
    s.pg /= s.mg;
  }
  const int per = (UP ? 4 : 1) * (int)sizeof(cplx) * s.pg * npar;  // bytes per coefficient
  s.mc = std::max(4, std::min(4 * nt, kShiftLds / per / 4 * 4));
  const size_t lds = std::max((size_t)per * s.mc, (size_t)(s.mg > 1 ? (UP ? 1 : 4) : 0) *
                                                      s.pg * (s.mg - 1) * s.rows * sizeof(cplx));
  const dim3 grid((unsigned)((ncols + s.pg * npar - 1) / (s.pg * npar)), (unsigned)s.tiles);
  const int4* sl = reinterpret_cast<const int4*>(slots);
  if (npar == 2)
    hipLaunchKernelGGL((k_shift<UP, SGN, 2>), grid, dim3(kShiftT), lds, st, ncols, nd, s, sh,
                       parents, sl, src, dst, A);
  else
    hipLaunchKernelGGL((k_shift<UP, SGN, 1>), grid, dim3(kShiftT), lds, st, ncols, nd, s, sh,
                       parents, sl, src, dst, A);
  hip_throw(hipGetLastError(), "shift");
}

}  // namespace fmm2d
