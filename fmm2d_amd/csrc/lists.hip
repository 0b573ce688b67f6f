// Interaction lists 1-4 (computelists, common/tree_routs2d.f:486-710).
//
// The reference builds them in one serial sweep that also appends to the
// lists of OTHER boxes (list1 and list4 of the finer neighbours of a leaf).
// Here every box gathers its own entries ("pull" form), so each box's
// thread writes only its own rows and no atomics are needed:
//   list2(b): children of the parent's colleagues not adjacent to b
//             (|dx| >= 1.05 bs or |dy| >= 1.05 bs, single-precision 1.05);
//   list1(b), leaf b: leaf colleagues (b included), children of non-leaf
//             colleagues that touch b, and coarser leaves (colleagues of b's
//             parent) that touch b;
//   list3(b), leaf b: children of non-leaf colleagues that do not touch b;
//   list4(b): coarser leaves among the parent's colleagues that do not
//             touch b.
// "Touch" uses distest = 1.05*(bs_l + bs_{l+1})/2 with strict <, as the
// reference.  Entries are the same sets as the reference's; their order
// within a row may differ (only summation order depends on it).
#include <algorithm>

#include "tree.h"

namespace fmm2d {
namespace {

constexpr double kColl = (double)1.05f;

// box size of every level, by value
constexpr int kListLevels = 54;
struct ListSizes {
  double v[kListLevels];
};

// One thread per box over the candidates (colleague k, child slot q) in order,
// so every row is in the order of a serial sweep.  Siblings are neighbouring
// threads and read the same boxes.  The loads of a sweep (nine colleagues, their
// children, their centres) do not depend on each other; a child's centre is
// formed from its parent's as the tree build does, not loaded.  The rows of M2L
// slots are assembled in LDS and written with consecutive threads on
// consecutive addresses.
// Three boxes a wavefront, with a lane for every two candidates and ranks by
// ballots, issued 230 wavefront instructions a box: 1.94e6 boxes 1.05 ms, this
// 0.20; 5e5 boxes 0.37 and 0.08.
constexpr int kListT = 128;

__global__ __launch_bounds__(kListT) void k_lists(
    int nb, const int* __restrict__ ilevel, const int* __restrict__ iparent,
    const int4* __restrict__ ichild, const int* __restrict__ ncoll, const int* __restrict__ coll,
    const double2* __restrict__ centers, ListSizes sz, int* n1, int* l1, int* n2, int* l2, int* n3,
    int* l3, int* n4, int* l4, int* s2) {
  __shared__ int slots[kListT * kSlots];
  __shared__ double bsl[kListLevels];
  const int tid = threadIdx.x;
  for (int k = tid; k < kListLevels; k += kListT) bsl[k] = sz.v[k];
  const int64_t b0 = xcd_block() * kListT;
  int* ssh = slots + tid * kSlots;
#pragma unroll
  for (int t = 0; t < kSlots; ++t) ssh[t] = -1;
  __syncthreads();
  const int64_t bb = b0 + tid;
  if (bb < nb) {
    const int b = (int)bb;
    const int lev = ilevel[b];
    const double2 c = centers[b];
    const int4 mine = ichild[b];
    int* r1 = l1 + (int64_t)kMaxList1 * b;
    int* r2 = l2 ? l2 + (int64_t)kMaxList2 * b : nullptr;
    int* r3 = l3 + (int64_t)kMaxList3 * b;
    int* r4 = l4 + (int64_t)kMaxList4 * b;
    int c1 = 0, c2 = 0, c3 = 0, c4 = 0;
    if (b == 0) {
      // the root: list 1 = itself when it is a leaf
      if (mine.x < 0) r1[c1++] = 0;
    } else {
      const int dad = iparent[b];
      const int4 sib = ichild[dad];
      const int qb = b == sib.x ? 0 : b == sib.y ? 1 : b == sib.z ? 2 : 3;  // child position
      int j[kMaxColl];
      int4 ch[kMaxColl];
      double2 cj[kMaxColl];
      auto load = [&](int box) {
        const int n = ncoll[box];
#pragma unroll
        for (int k = 0; k < kMaxColl; ++k) j[k] = coll[kMaxColl * (int64_t)box + k];
#pragma unroll
        for (int k = 0; k < kMaxColl; ++k) {
          if (k >= n) j[k] = -1;
          ch[k] = ichild[max(j[k], 0)];
          cj[k] = centers[max(j[k], 0)];
        }
      };
      load(dad);
      // list 2 from the children of the parent's colleagues, and their slots;
      // coarser leaves among the colleagues go to list 1 or 4
      const double lim = kColl * bsl[lev], binv = 1.0 / bsl[lev], h = 0.5 * bsl[lev];
      const double dist4 = lev >= 2 ? 1.05 * (bsl[lev - 1] + bsl[lev]) / 2.0 : 0.0;
#pragma unroll
      for (int k = 0; k < kMaxColl; ++k) {
        if (j[k] < 0) continue;
        if (ch[k].x < 0) {
          if (lev >= 2) {
            const double xd = fabs(cj[k].x - c.x), yd = fabs(cj[k].y - c.y);
            if (xd < dist4 && yd < dist4) {
              if (c1 < kMaxList1) r1[c1] = j[k];
              ++c1;
            } else {
              if (c4 < kMaxList4) r4[c4] = j[k];
              ++c4;
            }
          }
          continue;
        }
        const int id[4] = {ch[k].x, ch[k].y, ch[k].z, ch[k].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double dx = (cj[k].x + ((q & 1) ? h : -h)) - c.x;
          const double dy = (cj[k].y + ((q & 2) ? h : -h)) - c.y;
          if (fabs(dx) >= lim || fabs(dy) >= lim) {
            const int sl = m2l_slot(qb, (int)rint(dx * binv), (int)rint(dy * binv));
            if (sl >= 0) ssh[sl] = id[q];
            // (the rows of list 2 are for callers that export them: the M2L reads s2)
            if (l2 && c2 < kMaxList2) r2[c2] = id[q];
            ++c2;
          }
        }
      }
      // own entries of a leaf: a leaf colleague itself, or the children of a
      // non-leaf colleague
      if (mine.x < 0) {
        load(b);
        const double dist = 1.05 * (bsl[lev] + bsl[lev + 1]) / 2.0, hc = 0.5 * bsl[lev + 1];
#pragma unroll
        for (int k = 0; k < kMaxColl; ++k) {
          if (j[k] < 0) continue;
          if (ch[k].x < 0) {
            if (c1 < kMaxList1) r1[c1] = j[k];
            ++c1;
            continue;
          }
          const int id[4] = {ch[k].x, ch[k].y, ch[k].z, ch[k].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const double xd = fabs((cj[k].x + ((q & 1) ? hc : -hc)) - c.x);
            const double yd = fabs((cj[k].y + ((q & 2) ? hc : -hc)) - c.y);
            if (xd < dist && yd < dist) {
              if (c1 < kMaxList1) r1[c1] = id[q];
              ++c1;
            } else {
              if (c3 < kMaxList3) r3[c3] = id[q];
              ++c3;
            }
          }
        }
      }
    }
    n1[b] = min(c1, kMaxList1);
    n2[b] = min(c2, kMaxList2);
    n3[b] = min(c3, kMaxList3);
    n4[b] = min(c4, kMaxList4);
  }
  __syncthreads();
  const int64_t left = nb - b0;
  const int m = (int)(left < kListT ? (left > 0 ? left : 0) : kListT) * kSlots;
  for (int t = tid; t < m; t += kListT) s2[b0 * kSlots + t] = slots[t];
}
}  // namespace

void build_lists(const Tree& t, Lists& L, hipStream_t st, bool rows2) {
  const int nb = t.nboxes;
  L.n1.alloc(nb, st);
  L.n2.alloc(nb, st);
  L.n3.alloc(nb, st);
  L.n4.alloc(nb, st);
  L.l1.alloc((size_t)kMaxList1 * nb, st);
  if (rows2) L.l2.alloc((size_t)kMaxList2 * nb, st);
  L.l3.alloc((size_t)kMaxList3 * nb, st);
  L.l4.alloc((size_t)kMaxList4 * nb, st);
  L.s2.alloc((size_t)kSlots * nb, st);
  // boxsize per level, with one extra (finer) entry for the leaf test at the
  // deepest level, where computelists never reaches it (no non-leaf colleague)
  ListSizes sz{};
  if (t.boxsize.size() + 1 > (size_t)kListLevels) throw HipError{hipErrorInvalidValue, "levels"};
  for (size_t l = 0; l < t.boxsize.size(); ++l) sz.v[l] = t.boxsize[l];
  sz.v[t.boxsize.size()] = t.boxsize.back() / 2;
  if (nb > 0) {
    hipLaunchKernelGGL(k_lists, dim3(xcd_grid(ceil_div(nb, kListT))), dim3(kListT), 0, st, nb,
                       t.ilevel.p, t.iparent.p, reinterpret_cast<const int4*>(t.ichild.p),
                       t.ncoll.p, t.coll.p, reinterpret_cast<const double2*>(t.centers.p), sz,
                       L.n1.p, L.l1.p, L.n2.p, L.l2.p, L.n3.p, L.l3.p, L.n4.p, L.l4.p, L.s2.p);
    hip_throw(hipGetLastError(), "kernel launch");
  }
}

}  // namespace fmm2d
