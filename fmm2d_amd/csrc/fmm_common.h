// Pieces shared by the FMM drivers (Laplace/Cauchy and Helmholtz): point
// gather/scatter, leaf lookup, the child and list-2 work plans that feed the
// MFMA translate kernel, work counters, upload and stage timing.
//
// Everything here has internal linkage (anonymous namespace), so each driver
// translation unit carries its own copy of the kernels.
#pragma once

#include <algorithm>
#include <cstring>
#include <vector>

#include "devbuf.h"
#include "scan.h"
#include "tree.h"

namespace fmm2d {
namespace {

constexpr int kW = 64;  // wavefront size
constexpr int kOff = 7;  // offsets -3..3 per axis

FMM2D_HD cplx cpowi(cplx w, int k) {
  cplx r = mkc(1.0), b = w;
  while (k) {
    if (k & 1) r = r * b;
    b = b * b;
    k >>= 1;
  }
  return r;
}

__device__ __forceinline__ int npts_eval(int b, const int* sse, const int* tse, int ifpgh,
                                         int ifpght) {
  int n = 0;
  if (ifpgh > 0) n += sse[2 * b + 1] - sse[2 * b];
  if (ifpght > 0) n += tse[2 * b + 1] - tse[2 * b];
  return n;
}


// ---------------------------------------------------------- gather / scatter
__global__ void k_gather_xy(int64_t n, const int* perm, const double* xy, double* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int j = perm[i];
  out[2 * i] = xy[2 * (int64_t)j];
  out[2 * i + 1] = xy[2 * (int64_t)j + 1];
}

// cfmm2d, hfmm2d: points and densities copied as they are (absent: null).
__global__ void k_gather_dens(int64_t n, int nd, const int* perm, const double* xy, double* oxy,
                              const cplx* ch, cplx* och, const cplx* ds, cplx* ods,
                              const double* dv, double* odv) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t j = perm[i];
  oxy[2 * i] = xy[2 * j];
  oxy[2 * i + 1] = xy[2 * j + 1];
  for (int d = 0; d < nd; ++d) {
    if (ch) och[i * nd + d] = ch[j * nd + d];
    if (ds) ods[i * nd + d] = ds[j * nd + d];
  }
  if (dv)
    for (int k = 0; k < 2 * nd; ++k) odv[i * 2 * nd + k] = dv[j * 2 * nd + k];
}

// out[perm[i]] = in[i] for m values per point, potential, gradient and second
// derivatives (absent: null)
__global__ void k_scatter(int64_t n, const int* perm, int m0, const cplx* in0, cplx* out0, int m1,
                          const cplx* in1, cplx* out1, int m2, const cplx* in2, cplx* out2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t j = perm[i];
  for (int k = 0; k < m0; ++k) out0[j * m0 + k] = in0[i * m0 + k];
  if (out1)
    for (int k = 0; k < m1; ++k) out1[j * m1 + k] = in1[i * m1 + k];
  if (out2)
    for (int k = 0; k < m2; ++k) out2[j * m2 + k] = in2[i * m2 + k];
}

// ---------------------------------------------------------- near-field segments
// The sources a leaf interacts with directly (the boxes of its list 1,
// common/tree_routs2d.f:486-710) as a few contiguous ranges of the sorted
// sources: empty boxes dropped, ranges sorted by start and merged where one
// ends at the next one's start (sibling leaves are adjacent in the sorted
// order).  Row b of kSegRow int2: [0] = {sources in total, ranges}, then
// the ranges [s0, s1), then an end mark {0, 0} (every box has a row; that of
// a box with an empty list 1 holds no range).
constexpr int kSegRow = 16;
static_assert(kSegRow >= kMaxList1 + 2, "segment row holds the list-1 ranges and the end mark");

__global__ __launch_bounds__(256) void k_near_segs(int64_t nb, const int* n1, const int* l1,
                                                   const int* sse, int2* seg) {
  __shared__ int2 buf[256][kMaxList1];
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int c1 = n1[b];
  int2* r = buf[threadIdx.x];
  int m = 0;
  for (int k = 0; k < c1; ++k) {  // insertion sort by start
    const int c = l1[(int64_t)kMaxList1 * b + k];
    const int s0 = sse[2 * c], s1 = sse[2 * c + 1];
    if (s1 <= s0) continue;
    int q = m++;
    for (; q > 0 && r[q - 1].x > s0; --q) r[q] = r[q - 1];
    r[q] = make_int2(s0, s1);
  }
  int2* out = seg + (int64_t)kSegRow * b;
  int ns = 0, tot = 0;
  for (int k = 0; k < m;) {
    int2 s = r[k++];
    for (; k < m && r[k].x == s.y; ++k) s.y = r[k].y;
    out[1 + ns++] = s;
    tot += s.y - s.x;
  }
  out[1 + ns] = make_int2(0, 0);
  out[0] = make_int2(tot, ns);
}

// true when pred holds on every active lane of the wavefront
__device__ __forceinline__ bool wave_all(bool pred) { return __ballot(pred) == __ballot(1); }

// Walks the ranges of one segment row: current range [j, e) and the next
// one prefetched, advanced when the current one runs out.
struct SegCursor {
  const int2* row;
  int j, e, k, last;
  int2 nxt;
  __device__ __forceinline__ int init(const int2* r) {
    row = r;
    const int2 hd = r[0];
    last = hd.y + 1;  // slot of the end mark
    const int2 cur = r[1];
    nxt = r[min(2, last)];
    k = 3;
    j = cur.x;
    e = cur.y;
    return hd.x;
  }
  __device__ __forceinline__ void step() {
    if (j == e) {
      j = nxt.x;
      e = nxt.y;
      nxt = row[min(k, last)];
      ++k;
    }
  }
};


// ---------------------------------------------------------- list-2 plan
// The M2L of one target box is sum over its list-2 sources of T_o M_c, with o
// the source's offset.  For a target in child position q of its parent the
// possible offsets form a fixed set of 27 (the 6x6 children of the parent's
// 3x3 neighbourhood minus the 3x3 adjacent ones), so targets of the same q are
// processed together by the translate kernel, one offset slot after another.
__device__ __forceinline__ bool m2l_target(int b, const int* ilevel, const int* n2, const int* sse,
                                           const int* tse, int ifpgh, int ifpght) {
  return ilevel[b] >= 2 && n2[b] > 0 && npts_eval(b, sse, tse, ifpgh, ifpght) > 0;
}

// A tree has 1 + 4 np boxes, np of them with children, and the boxes of a level
// l >= 1 are groups of four siblings: the k-th group of level l + 1 belongs to
// a non-leaf box of level l, so the groups number the non-leaf boxes level by
// level (pos[l] = groups of the levels up to l) and no list has to be made.
constexpr int kPlanLevels = 54;
struct PlanLevels {
  int nl;
  int lstart[kPlanLevels], pos[kPlanLevels];
};

// For the non-leaf box of group i: its id (list), the child slots of M2M (up: a
// child without sources is skipped, laprouts2d.f via cfmm2d.f:962-983) and
// L2L (down: all children when the parent has points to evaluate,
// cfmm2d.f:1042-1076), and the child in position q if it is an M2L target
// (tl[q np + i], else -1): siblings sit at the same position of the four
// classes.  With p2l, also the boxes with list-4 work, in any order (their
// number in *np2l, zero before).
constexpr int kPlanT = 1024;
__global__ __launch_bounds__(kPlanT) void k_plan(int64_t nb, int np, PlanLevels T, const int* iparent, const int* ilevel,
                       const int* n2, const int* n4, const int* sse, const int* tse, int ifpgh,
                       int ifpght, int* list, int* up, int* down, int* tl, int* p2l,
                       int* np2l) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) {
    int l = 0;
    while (l + 1 < T.nl && T.pos[l + 1] <= i) ++l;
    const int c0 = T.lstart[l + 1] + 4 * ((int)i - T.pos[l]);
    const int b = iparent[c0];
    const bool ev = npts_eval(b, sse, tse, ifpgh, ifpght) > 0;
    list[i] = b;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = c0 + q;
      up[4 * i + q] = (sse[2 * c + 1] > sse[2 * c]) ? c : -1;
      down[4 * i + q] = ev ? c : -1;
      tl[(int64_t)q * np + i] = m2l_target(c, ilevel, n2, sse, tse, ifpgh, ifpght) ? c : -1;
    }
  }
  if (p2l) {
    const bool f = i < nb && ilevel[i] >= 2 && n4[i] > 0 &&
                   npts_eval((int)i, sse, tse, ifpgh, ifpght) > 0;
    // one atomic a workgroup: one a wavefront took 0.2 ms for 6e5 boxes
    __shared__ int wcnt[kPlanT / 64], base;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long m = __ballot(f);
    if (lane == 0) wcnt[w] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
      int s = 0;
      for (int k = 0; k < kPlanT / 64; ++k) s += wcnt[k];
      base = s ? atomicAdd(np2l, s) : 0;
    }
    __syncthreads();
    int at = base + __popcll(m & ((1ull << lane) - 1ull));
    for (int k = 0; k < w; ++k) at += wcnt[k];
    if (f) p2l[at] = (int)i;
  }
}

// ---------------------------------------------------------- work counters
// cnt[0] near pairs, [1] list-2 pairs, [2] M2M edges, [3] L2L edges,
// [4] list-3 (point, box) pairs, [5] list-4 (source, box) pairs; M2M edges
// count at the parent, L2L edges at the child.  These are the edges of the
// reference's algorithm, whose upward and downward passes reach level 1; the
// drivers leave the parents of levels 0 and 1 out, whose expansions nothing reads.
__global__ void k_counts(int64_t n, const int* ilevel, const int* iparent, const int* nchild,
                         const int* ichild, const int* sse, const int* tse, int ifpgh,
                         int ifpght, const int* n1, const int* l1, const int* n2, const int* n3,
                         const int* n4, const int* l4, int b0, unsigned long long* cnt) {
  // boxes b0 .. b0+n-1; cnt is the same for every lane, so the compiler
  // combines each wavefront's atomics into one
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = b0 + (int)i;
  const int lev = ilevel[b];
  const int ne = npts_eval(b, sse, tse, ifpgh, ifpght);
  unsigned long long near = 0, l3 = 0, l4c = 0, m2m = 0, l2l = 0, m2l = 0;
  if (nchild[b] == 0) {
    unsigned long long s = 0;
    for (int k = 0; k < n1[b]; ++k) {
      const int c = l1[(int64_t)kMaxList1 * b + k];
      s += sse[2 * c + 1] - sse[2 * c];
    }
    near = s * (unsigned long long)ne;
    l3 = (unsigned long long)n3[b] * ne;
  } else if (lev >= 1) {
    for (int q = 0; q < 4; ++q) {
      const int c = ichild[4 * b + q];
      if (sse[2 * c + 1] > sse[2 * c]) ++m2m;
    }
  }
  if (lev >= 2 && ne > 0) {
    m2l = n2[b];
    for (int k = 0; k < n4[b]; ++k) {
      const int c = l4[(int64_t)kMaxList4 * b + k];
      l4c += sse[2 * c + 1] - sse[2 * c];
    }
    if (npts_eval(iparent[b], sse, tse, ifpgh, ifpght) > 0) l2l = 1;
  }
  if (near) atomicAdd(&cnt[0], near);
  if (m2l) atomicAdd(&cnt[1], m2l);
  if (m2m) atomicAdd(&cnt[2], m2m);
  if (l2l) atomicAdd(&cnt[3], l2l);
  if (l3) atomicAdd(&cnt[4], l3);
  if (l4c) atomicAdd(&cnt[5], l4c);
}


template <typename T> DBuf<T> upload(const std::vector<T>& v, hipStream_t st) {
  static_assert(sizeof(T) % 4 == 0, "upload_bytes moves 4-byte words");
  DBuf<T> d(v.size(), st);
  upload_bytes(d.p, v.data(), sizeof(T) * v.size(), st);  // v may die after return
  return d;
}


struct Timer {
  bool on;
  hipStream_t st;
  std::vector<hipEvent_t> ev;
  std::vector<int> slot;
  Timer(bool enable, hipStream_t s) : on(enable), st(s) { mark(-1); }
  void mark(int s) {
    if (!on) return;
    hipEvent_t e;
    // (without the system-scope fence of the default: 2.7 us a mark, not 4)
    (void)hipEventCreateWithFlags(&e, hipEventDisableSystemFence);
    (void)hipEventRecord(e, st);
    ev.push_back(e);
    slot.push_back(s);
  }
  // after a stream sync: accumulate interval k (ending at event k) into slot
  void collect(double* out) {
    if (!on) return;
    for (size_t k = 1; k < ev.size(); ++k) {
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, ev[k - 1], ev[k]);
      if (slot[k] >= 0) out[slot[k]] += 1e-3 * ms;
    }
    float tot = 0.f;
    (void)hipEventElapsedTime(&tot, ev.front(), ev.back());
    out[11] = 1e-3 * tot;
  }
  ~Timer() {
    for (auto e : ev) (void)hipEventDestroy(e);
  }
};


// The work lists of k_plan.  list[lev_pos[l] .. lev_pos[l+1]) are the non-leaf
// boxes of level l; the M2L targets of level l in child position q are tl[q np
// + lev_pos[l-1] .. q np + lev_pos[l]).
struct BoxPlan {
  DBuf<int> list, up, down, tl, p2l;
  std::vector<int> lev_pos;
  int np = 0;
};

// np2l: a zeroed device counter, or null when the list-4 boxes are not needed
void plan_boxes(const Tree& t, const Lists& L, int pg, int pgt, BoxPlan& bp, int* np2l,
                hipStream_t st) {
  const int nb = t.nboxes, nl = t.nlevels;
  PlanLevels T{};
  T.nl = nl;
  if (nl + 2 > kPlanLevels) throw HipError{hipErrorInvalidValue, "tree levels"};
  bp.lev_pos.assign(nl + 2, 0);
  for (int l = 0; l <= nl; ++l) {
    T.lstart[l] = t.lstart[l];
    T.pos[l] = bp.lev_pos[l];
    const int next = l < nl ? (l + 1 < nl ? t.lstart[l + 2] : nb) - t.lstart[l + 1] : 0;
    bp.lev_pos[l + 1] = bp.lev_pos[l] + next / 4;
  }
  bp.np = bp.lev_pos[nl + 1];
  const size_t np = (size_t)std::max(bp.np, 1);
  bp.list.alloc(np, st);
  bp.up.alloc(4 * np, st);
  bp.down.alloc(4 * np, st);
  bp.tl.alloc(4 * np, st);
  if (np2l) bp.p2l.alloc(nb, st);
  hipLaunchKernelGGL(k_plan, dim3((unsigned)((nb + kPlanT - 1) / kPlanT)), dim3(kPlanT), 0, st,
                     (int64_t)nb, bp.np, T, t.iparent.p, t.ilevel.p, L.n2.p, L.n4.p, t.isrcse.p,
                     t.itargse.p, pg, pgt, bp.list.p, bp.up.p, bp.down.p, bp.tl.p, bp.p2l.p, np2l);
  hip_throw(hipGetLastError(), "plan");
}

// Several small host arrays in one upload.
struct Blob {
  std::vector<unsigned> w;
  DBuf<unsigned> d;
  template <typename T> size_t add(const std::vector<T>& v) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    const size_t at = (w.size() + 3) & ~size_t(3);
    w.resize(at + v.size() * (sizeof(T) / 4), 0u);
    if (!v.empty()) std::memcpy(w.data() + at, v.data(), v.size() * sizeof(T));
    return at;
  }
  void upload(hipStream_t st) {
    d.alloc(w.size(), st);
    upload_bytes(d.p, w.data(), 4 * w.size(), st);
  }
  template <typename T> T* at(size_t off) const { return reinterpret_cast<T*>(d.p + off); }
};

// slot -> offset index (dx+3)*7 + (dy+3) for each child position q
std::vector<int> m2l_slot_offsets() {
  std::vector<int> soff(4 * kSlots, 0);
  for (int q = 0; q < 4; ++q)
    for (int dx = -3; dx <= 3; ++dx)
      for (int dy = -3; dy <= 3; ++dy) {
        const int sl = m2l_slot(q, dx, dy);
        if (sl >= 0) soff[q * kSlots + sl] = (dx + 3) * kOff + (dy + 3);
      }
  return soff;
}

}  // namespace
}  // namespace fmm2d
