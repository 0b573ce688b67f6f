// Adaptive quadtree built on the GPU, box-for-box identical to the reference.
//
// Reference (common/pts_tree2d.f, common/tree_routs2d.f):
//   pts_tree_build 406-655   level-by-level refinement of boxes holding more
//                            than ndiv points, 4 children each, numbered in
//                            parent order (tree_refine_boxes 9-56)
//   computecoll 100-211      colleagues: same-level boxes with centres within
//                            1.05*bs (a single-precision 1.05, promoted)
//   pts_tree_fix_lr 758-1061 level restriction: flag / flag+ passes, refine,
//                            reorganise, then flag++ (updateflags 217-326)
//   pts_tree_reorg 1066-1215 per level: original boxes first, then new ones
//   pts_tree_sort 1222-1246  stable recursive partition of the points
//
// GPU formulation: one thread per point for classification into children
// (y - cy < 0 then x - cx < 0, as sort_pts_to_children 659-754), one thread
// per box for every box-level step, device prefix sums (scan.h) where the
// reference uses cumsum, and the final point order as the points of each leaf (a contiguous
// range of the path order) in input order -- which is exactly the order the
// reference's recursive stable partition produces.  Box-level steps run level
// by level where the reference's loops carry a dependency between levels.

#include <algorithm>
#include <cmath>
#include <memory>

#include "radix_sort.h"
#include "scan.h"
#include "tree.h"

namespace fmm2d {
namespace {

// The reference writes `1.05*boxsize(ilev)` with a default-real literal in
// computecoll / computelists: 1.05 rounded to single precision, then promoted.
constexpr double kColl = (double)1.05f;
constexpr int kMaxLevels = 51;  // nlmax of the reference (pts_tree2d.f)
constexpr int kBatch = 8;             // refinement levels per host synchronisation
constexpr int64_t kBatchBoxes = 1 << 24;  // box capacity a batch may reserve

// copy the first n[k] 4-byte words of src[k] to dst[k] for k = blockIdx.y
struct WordCopies {
  const unsigned* src[8];
  unsigned* dst[8];
  int64_t n[8];
};
__global__ void k_copy_words(WordCopies c) {
  const int k = blockIdx.y;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < c.n[k];
       i += (int64_t)gridDim.x * blockDim.x)
    c.dst[k][i] = c.src[k][i];
}

// The arrays that describe cap boxes.  The colleagues, 40 of a box's 104 bytes,
// come with the first search for them and for the boxes there are then: the
// refinement reserves more boxes than it makes.
struct Boxes {
  DBuf<double> centers;
  DBuf<int> ilevel, iparent, nchild, ichild, ses, set, iflag;
  DBuf<int> ncoll, coll;
  size_t cap = 0;
  void alloc(size_t c, hipStream_t st) {
    cap = c;
    centers.alloc(2 * c, st);
    ilevel.alloc(c, st);
    iparent.alloc(c, st);
    nchild.alloc(c, st);
    ichild.alloc(4 * c, st);
    ses.alloc(2 * c, st);
    set.alloc(2 * c, st);
    iflag.alloc(c, st);
  }
  // room for the colleagues of c boxes (contents lost if there was less)
  void alloc_coll(size_t c) {
    if (ncoll.n >= c) return;
    coll.reset();
    ncoll.alloc(c, ilevel.st);
    coll.alloc(kMaxColl * c, ilevel.st);
  }
  void swap_boxes(Boxes& o) {
    centers.swap(o.centers);
    ilevel.swap(o.ilevel);
    iparent.swap(o.iparent);
    nchild.swap(o.nchild);
    ichild.swap(o.ichild);
    ses.swap(o.ses);
    set.swap(o.set);
    iflag.swap(o.iflag);
    std::swap(cap, o.cap);
  }
  // capacity for `need` boxes, the first `keep` kept (one copy launch)
  void fit(size_t need, size_t keep) {
    if (need <= cap) return;
    const hipStream_t st = ilevel.st;
    Boxes b;
    b.alloc(need, st);
    if (keep > 0) {
      WordCopies c{};
      int k = 0;
      auto add = [&](const void* from, void* to, size_t words) {
        c.src[k] = static_cast<const unsigned*>(from);
        c.dst[k] = static_cast<unsigned*>(to);
        c.n[k++] = (int64_t)words;
      };
      add(centers.p, b.centers.p, 4 * keep);  // 2 doubles per box
      add(ilevel.p, b.ilevel.p, keep);
      add(iparent.p, b.iparent.p, keep);
      add(nchild.p, b.nchild.p, keep);
      add(ichild.p, b.ichild.p, 4 * keep);
      add(ses.p, b.ses.p, 2 * keep);
      add(set.p, b.set.p, 2 * keep);
      add(iflag.p, b.iflag.p, keep);
      const unsigned gx = (unsigned)std::min<int64_t>(ceil_div((int64_t)(4 * keep), 256), 1024);
      hipLaunchKernelGGL(k_copy_words, dim3(gx, 8), dim3(256), 0, st, c);
      hip_throw(hipGetLastError(), "box copy");
    }
    swap_boxes(b);
  }
  // the same with twice the capacity there was, for boxes that come level by level
  void grow(size_t need, size_t keep) {
    if (need > cap) fit(std::max(need, 2 * cap), keep);
  }
};

// ------------------------------------------------------------ bounding box
// min, max, min, max over a workgroup of NW waves, on every thread
template <int NW>
__device__ __forceinline__ void block_bounds(double* v, double (*sm)[4]) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    v[0] = fmin(v[0], __shfl_xor(v[0], d, 64));
    v[1] = fmax(v[1], __shfl_xor(v[1], d, 64));
    v[2] = fmin(v[2], __shfl_xor(v[2], d, 64));
    v[3] = fmax(v[3], __shfl_xor(v[3], d, 64));
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 4; ++k) sm[w][k] = v[k];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    v[0] = fmin(v[0], sm[i][0]);
    v[1] = fmax(v[1], sm[i][1]);
    v[2] = fmin(v[2], sm[i][2]);
    v[3] = fmax(v[3], sm[i][3]);
  }
}

constexpr int kRedBlocks = 512;

// Per-block bounds of all points into part[4 block ..]; also clears the words
// that the key kernel and the sort count in.
__global__ __launch_bounds__(256) void k_bbox_partial(const double* __restrict__ src, int64_t ns,
                                                      const double* __restrict__ trg, int64_t nt,
                                                      double* part, unsigned* words,
                                                      int64_t nwords) {
  __shared__ double sm[4][4];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nwords;
       i += (int64_t)gridDim.x * 256)
    words[i] = 0;
  double v[4] = {INFINITY, -INFINITY, INFINITY, -INFINITY};
  const int64_t n = ns + nt;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double* p = (i < ns) ? (src + 2 * i) : (trg + 2 * (i - ns));
    double x = p[0], y = p[1];
    v[0] = fmin(v[0], x);
    v[1] = fmax(v[1], x);
    v[2] = fmin(v[2], y);
    v[3] = fmax(v[3], y);
  }
  block_bounds<4>(v, sm);
  if (threadIdx.x == 0)
    for (int k = 0; k < 4; ++k) part[4 * blockIdx.x + k] = v[k];
}

// The bounds from the per-block ones, by every workgroup that needs them
// (at most 16 KiB of L2 reads), into v on every thread.
template <int NW>
__device__ __forceinline__ void bounds_of_parts(const double* part, int nb, double* v,
                                                double (*sm)[4]) {
  v[0] = v[2] = INFINITY;
  v[1] = v[3] = -INFINITY;
  for (int i = threadIdx.x; i < nb; i += 64 * NW) {
    v[0] = fmin(v[0], part[4 * i]);
    v[1] = fmax(v[1], part[4 * i + 1]);
    v[2] = fmin(v[2], part[4 * i + 2]);
    v[3] = fmax(v[3], part[4 * i + 3]);
  }
  block_bounds<NW>(v, sm);
}

// Bounding square (pts_tree2d.f:455-517) of the bounds
FMM2D_HD void root_square(const double* bb, double* cx, double* cy, double* bs) {
  *bs = bb[1] - bb[0];
  const double sizey = bb[3] - bb[2];
  if (sizey > *bs) *bs = sizey;
  *cx = (bb[0] + bb[1]) / 2;
  *cy = (bb[2] + bb[3]) / 2;
}

// ------------------------------------------------------------ point paths
// Each point's path through the tree is the sequence of its quadrants,
// computed with the reference's own centre arithmetic: child centre = parent
// centre +- bs_child/2 (one rounding), point below/left of the centre when
// y - cy < 0 / x - cx < 0.  The path does not depend on which boxes get
// refined, so it is computed once per point; digits are child indices 0..3 in
// the reference's order (1=(-,-), 2=(+,-), 3=(-,+), 4=(+,+)), most significant
// digit = level 1.  Levels 1..20 go to key1 (a 40-bit radix sort), levels
// 21..51 to key2 (only computed when the tree is that deep).  x - cx < 0 is
// tested as x < cx: with gradual underflow the difference of two distinct
// finite doubles is never rounded to zero and keeps its sign, and both forms
// are false for NaN.
constexpr int kD1 = 20;
constexpr int kD2Max = 31;

// The path of (x, y) over `levels` levels from the box (cx, cy) of half size
// 2 h on, which moves along (box sizes are halved exactly as the reference's
// boxsize(l+1) = boxsize(l)/2).
__device__ __forceinline__ unsigned long long path_key(double x, double y, double& cx, double& cy,
                                                       double& h, int levels) {
  unsigned long long k = 0;
  for (int l = 0; l < levels; ++l) {
    const int qx = (x < cx) ? 0 : 1, qy = (y < cy) ? 0 : 1;
    k = (k << 2) | (unsigned long long)(2 * qy + qx);
    h *= 0.5;
    cx += qx ? h : -h;
    cy += qy ? h : -h;
  }
  return k;
}

// The keys of one set over d1 and (second word) d2 further levels
__global__ void k_path_keys(int64_t n, const double* __restrict__ xy, double cx0, double cy0,
                            double bs0, int d1, int d2, unsigned long long* key1,
                            unsigned long long* key2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double cx = cx0, cy = cy0, h = 0.5 * bs0;
  key1[i] = path_key(xy[2 * i], xy[2 * i + 1], cx, cy, h, d1);
  key2[i] = path_key(xy[2 * i], xy[2 * i + 1], cx, cy, h, d2);
}

// The keys of d1 levels of both sets (blockIdx.y), from the per-block bounds,
// with the digit counts of their sort (hist[set][pass][digit]); block 0
// writes the bounds.
__global__ __launch_bounds__(kRsCountThreads) void k_keys_count(const double* __restrict__ src, int64_t ns,
                                                    const double* __restrict__ trg, int64_t nt,
                                                    const double* part, int nb, int d1,
                                                    int npass, unsigned long long* ksrc,
                                                    unsigned long long* ktrg, unsigned* hist,
                                                    double* bounds) {
  constexpr int kP = (2 * kD1 + 7) / 8;
  constexpr int NT = kRsCountThreads;
  __shared__ double sm[NT / 64][4];
  __shared__ unsigned h[kP][256];
  double bb[4];
  bounds_of_parts<NT / 64>(part, nb, bb, sm);
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0)
    for (int k = 0; k < 4; ++k) bounds[k] = bb[k];
  for (int q = threadIdx.x; q < kP * 256; q += NT) (&h[0][0])[q] = 0;
  __syncthreads();
  const double* xy = blockIdx.y ? trg : src;
  const int64_t n = blockIdx.y ? nt : ns;
  unsigned long long* out = blockIdx.y ? ktrg : ksrc;
  double cx0, cy0, bs0;
  root_square(bb, &cx0, &cy0, &bs0);
  for (int64_t i0 = (int64_t)blockIdx.x * NT; i0 < n; i0 += (int64_t)gridDim.x * NT) {
    const int64_t i = i0 + threadIdx.x;
    unsigned long long k = 0;
    if (i < n) {
      double cx = cx0, cy = cy0, hh = 0.5 * bs0;
      k = path_key(xy[2 * i], xy[2 * i + 1], cx, cy, hh, d1);
      out[i] = k;
    }
    rs_count<kP>(h, k, i < n, npass);
  }
  __syncthreads();
  hist += (size_t)256 * npass * blockIdx.y;
  for (int q = threadIdx.x; q < npass * 256; q += NT)
    if ((&h[0][0])[q]) atomicAdd(&hist[q], (&h[0][0])[q]);
}

template <typename T>
__global__ void k_gather_by(int64_t n, const int* idx, const T* in, T* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = in[idx[i]];
}

struct Keys {
  const unsigned long long* k1;
  const unsigned long long* k2;  // null unless the tree is deeper than kD1
  int d1, d2;
};

__device__ __forceinline__ int digit_at(const Keys& K, int64_t i, int lev) {
  if (lev <= K.d1) return (int)((K.k1[i] >> (2 * (K.d1 - lev))) & 3ull);
  return (int)((K.k2[i] >> (2 * (K.d2 - (lev - K.d1)))) & 3ull);
}

// b[q] = first i in [lo0, hi0) whose digit at level lev is >= q + 1, q = 0..2
// (digits are sorted there because all keys in a box's range share the path
// above lev).  The three binary searches run interleaved over the whole
// range with their loads in flight together: at the first levels a box holds
// millions of points, and chained searches were ~60 dependent loads long.
__device__ void digit_bounds3(const Keys& K, int64_t lo0, int64_t hi0, int lev, int64_t* b) {
  int64_t lo[3] = {lo0, lo0, lo0}, hi[3] = {hi0, hi0, hi0};
  while (lo[0] < hi[0] || lo[1] < hi[1] || lo[2] < hi[2]) {
    int64_t mid[3];
    int dg[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) mid[q] = min(lo[q] + ((hi[q] - lo[q]) >> 1), hi0 - 1);
#pragma unroll
    for (int q = 0; q < 3; ++q) dg[q] = digit_at(K, mid[q], lev);  // lo0 <= mid < hi0
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      if (lo[q] < hi[q]) {
        if (dg[q] < q + 1) lo[q] = mid[q] + 1;
        else hi[q] = mid[q];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) b[q] = lo[q];
}

// ------------------------------------------------------------ refinement
__global__ void k_refine_flags(int64_t n, int lo, const int* ses, const int* set, int idivflag,
                               int ndiv, int* flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = lo + (int)i;
  const int cs = ses[2 * b + 1] - ses[2 * b], ct = set[2 * b + 1] - set[2 * b];
  int nn = cs;
  if (idivflag == 1) nn = ct;
  if (idivflag == 2) nn = max(cs, ct);
  flag[i] = nn > ndiv ? 1 : 0;
}

// *total = flags set in flag[0..n), from its exclusive scan offs
__global__ void k_total(int n, const int* flag, const int* offs, int* total) {
  *total = (n > 0) ? offs[n - 1] + flag[n - 1] : 0;
}

// Refinement of several levels between host synchronisations: dlev[2 l],
// dlev[2 l + 1] hold the first box and the box count of level l, the launches
// cover an upper bound of the level's size and read the count from dlev.  Two
// launches a level: the full boxes of every 256 (part), then their children,
// each workgroup adding the counts of those before it; the last one of the
// level writes the next level's range.
constexpr int kRefTile = 256;

__device__ __forceinline__ bool box_full(int b, const int* ses, const int* set, int idivflag,
                                         int ndiv) {
  const int cs = ses[2 * b + 1] - ses[2 * b], ct = set[2 * b + 1] - set[2 * b];
  int nn = cs;
  if (idivflag == 1) nn = ct;
  if (idivflag == 2) nn = max(cs, ct);
  return nn > ndiv;
}

__global__ __launch_bounds__(kRefTile) void k_lv_count(const int* dlev, int l, const int* ses,
                                                       const int* set, int idivflag, int ndiv,
                                                       int* part) {
  const int lo = dlev[2 * l], n = dlev[2 * l + 1];
  const int64_t i = (int64_t)blockIdx.x * kRefTile + threadIdx.x;
  if ((int64_t)blockIdx.x * kRefTile >= n) return;
  const int c = __syncthreads_count(i < n && box_full(lo + (int)i, ses, set, idivflag, ndiv));
  if (threadIdx.x == 0) part[blockIdx.x] = c;
}

// the sum of part[0 .. m), on every thread of a workgroup of 256
__device__ __forceinline__ int sum_parts(const int* part, int m, int* lds) {
  int s = 0, tot;
  for (int k = threadIdx.x; k < m; k += kRefTile) s += part[k];
  block_exclusive_scan(s, lds, &tot);
  return tot;
}

// Children of the flagged boxes lo..lo+n-1 are numbered base + 4*offs + q, q =
// 0..3 for (-,-), (+,-), (-,+), (+,+) around the parent centre
// (tree_refine_boxes, tree_routs2d.f:25-52).  Their point ranges split the
// parent's by the path digit at level lev.  mode 1 (level-restriction
// refinement): child iflag = 3 when the parent's flag is 1, else 0.
// the four children of box b, numbered c0 .. c0+3, at level lev
__device__ void make_children_of(int b, int c0, double half, int lev, double* centers,
                                 int* ilevel, int* iparent, int* nchild, int* ichild, int* ses,
                                 int* set, int* iflag, int mode, const Keys& ks,
                                 const Keys& kt) {
  const double cx = centers[2 * b], cy = centers[2 * b + 1];
  nchild[b] = 4;
  const int pf = (mode == 1) ? iflag[b] : 0;
  int bs_[5], bt_[5];
  bs_[0] = ses[2 * b];
  bs_[4] = ses[2 * b + 1];
  bt_[0] = set[2 * b];
  bt_[4] = set[2 * b + 1];
  int64_t bq[3];
  digit_bounds3(ks, bs_[0], bs_[4], lev, bq);
  for (int q = 1; q < 4; ++q) bs_[q] = (int)bq[q - 1];
  digit_bounds3(kt, bt_[0], bt_[4], lev, bq);
  for (int q = 1; q < 4; ++q) bt_[q] = (int)bq[q - 1];
  for (int q = 0; q < 4; ++q) {
    const int c = c0 + q;
    centers[2 * c] = cx + ((q & 1) ? half : -half);
    centers[2 * c + 1] = cy + ((q & 2) ? half : -half);
    iparent[c] = b;
    nchild[c] = 0;
    ichild[4 * c] = ichild[4 * c + 1] = ichild[4 * c + 2] = ichild[4 * c + 3] = -1;
    ichild[4 * b + q] = c;
    ilevel[c] = lev;
    ses[2 * c] = bs_[q];
    ses[2 * c + 1] = bs_[q + 1];
    set[2 * c] = bt_[q];
    set[2 * c + 1] = bt_[q + 1];
    iflag[c] = (mode == 1 && pf == 1) ? 3 : 0;
  }
}

__global__ void k_make_children(int64_t n, int lo, const int* flag, const int* offs, int base,
                                double half, int lev, double* centers, int* ilevel, int* iparent,
                                int* nchild, int* ichild, int* ses, int* set, int* iflag, int mode,
                                Keys ks, Keys kt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !flag[i]) return;
  make_children_of(lo + (int)i, base + 4 * offs[i], half, lev, centers, ilevel, iparent, nchild,
                   ichild, ses, set, iflag, mode, ks, kt);
}

__global__ __launch_bounds__(kRefTile) void k_lv_children(int* dlev, int l, const int* part,
                                                          int idivflag, int ndiv, double half,
                                                          double* centers, int* ilevel,
                                                          int* iparent, int* nchild, int* ichild,
                                                          int* ses, int* set, int* iflag, Keys ks,
                                                          Keys kt) {
  __shared__ int lds[kScanWaves + 1];
  const int lo = dlev[2 * l], n = dlev[2 * l + 1];
  const int64_t i0 = (int64_t)blockIdx.x * kRefTile, i = i0 + threadIdx.x;
  const int nb = lo + n;  // the level's boxes are the last ones made
  if (i0 >= n) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      dlev[2 * (l + 1)] = nb;
      dlev[2 * (l + 1) + 1] = 0;
    }
    return;
  }
  const int carry = sum_parts(part, blockIdx.x, lds);
  const bool f = i < n && box_full(lo + (int)i, ses, set, idivflag, ndiv);
  int own;
  const int ex = block_exclusive_scan(f ? 1 : 0, lds, &own);
  if (i0 + kRefTile >= n && threadIdx.x == 0) {
    dlev[2 * (l + 1)] = nb;
    dlev[2 * (l + 1) + 1] = 4 * (carry + own);
  }
  if (f)
    make_children_of(lo + (int)i, nb + 4 * (carry + ex), half, l + 1, centers, ilevel, iparent,
                     nchild, ichild, ses, set, iflag, 0, ks, kt);
}

// ------------------------------------------------------------ colleagues
// computecoll (tree_routs2d.f:100-211) for boxes lo..lo+n-1 of one level.
__global__ void k_coll(int64_t n, int lo, double bs, const int* iparent, const int* ichild,
                       const double* centers, int* ncoll, int* coll) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = lo + (int)i;
  const int dad = iparent[b];
  const double cx = centers[2 * b], cy = centers[2 * b + 1];
  const double lim = kColl * bs;
  int cnt = 0;
  const int nd = ncoll[dad];
  for (int k = 0; k < nd; ++k) {
    const int j = coll[9 * dad + k];
    for (int q = 0; q < 4; ++q) {
      const int kb = ichild[4 * j + q];
      if (kb >= 0 && fabs(centers[2 * kb] - cx) <= lim && fabs(centers[2 * kb + 1] - cy) <= lim) {
        if (cnt < kMaxColl) coll[9 * b + cnt] = kb;
        ++cnt;
      }
    }
  }
  ncoll[b] = min(cnt, kMaxColl);
  for (int k = cnt; k < kMaxColl; ++k) coll[9 * b + k] = -1;
}

// computecoll for every box at once (trees of at most kWalkLevels levels).
// The colleagues of a box are the boxes of its level whose integer
// coordinates (ix, iy) differ by at most one in each direction -- exactly the
// boxes the reference finds among the children of the parent's colleagues
// within 1.05 box sizes.  The reference lists them in the order of the
// parent's colleagues and then of the child slots (-,-), (+,-), (-,+), (+,+),
// which, by induction from the root, is increasing path order: the
// interleaved code of (iy, ix), iy bit above ix bit, coarsest level first.
constexpr int kWalkLevels = 29;

// spread the 29 bits of v to the even bit positions
__device__ __forceinline__ unsigned long long spread_bits(unsigned v) {
  unsigned long long x = v;
  x = (x | (x << 16)) & 0x0000FFFF0000FFFFull;
  x = (x | (x << 8)) & 0x00FF00FF00FF00FFull;
  x = (x | (x << 4)) & 0x0F0F0F0F0F0F0F0Full;
  x = (x | (x << 2)) & 0x3333333333333333ull;
  x = (x | (x << 1)) & 0x5555555555555555ull;
  return x;
}

// interleaved path code of (ix, iy) at one level, iy bit above ix bit
__device__ __forceinline__ unsigned long long path_code(unsigned ix, unsigned iy) {
  return spread_bits(ix) | (spread_bits(iy) << 1);
}

// Colleagues of every box in one pass.  A box's coordinates (ix, iy) come from
// walking up to the root: the child centre is the parent centre +- half the
// child size, so the comparisons are exact.  The neighbour (jx, jy) of box b
// (level lev) shares b's ancestors down to level
// m = lev - max(bitlength(ix ^ jx), bitlength(iy ^ jy)); it is found by going
// up lev - m parents and down lev - m child slots, slot 2 qy + qx taken from
// the bits of (jx, jy) (the reference's child order (-,-), (+,-), (-,+),
// (+,+)); a missing child ends the search.  Sets *big (if given) where a leaf
// holds more than big_max sources or targets.
__global__ void k_coll_walk(int64_t nb, const int* ilevel, const int* iparent, const int* ichild,
                            const double* centers, int* ncoll, int* coll, const int* nchild,
                            const int* ses, const int* set, int big_max, int* big) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb) return;
  const int b = (int)i;
  const int lev = ilevel[b];
  if (big && nchild[b] == 0) {
    const int m = max(ses[2 * i + 1] - ses[2 * i], set[2 * i + 1] - set[2 * i]);
    if (m > big_max) *big = 1;
  }
  const long long side = 1ll << lev;
  unsigned ix = 0, iy = 0;
  {
    int cur = b;
    double cx = centers[2 * cur], cy = centers[2 * cur + 1];
    for (int t = 0; t < lev; ++t) {
      const int par = iparent[cur];
      const double px = centers[2 * par], py = centers[2 * par + 1];
      ix |= (cx > px ? 1u : 0u) << t;
      iy |= (cy > py ? 1u : 0u) << t;
      cur = par;
      cx = px;
      cy = py;
    }
  }
  int id[kMaxColl];
  unsigned long long code[kMaxColl];
  int cnt = 0;
  for (int dy = -1; dy <= 1; ++dy)
    for (int dx = -1; dx <= 1; ++dx) {
      const long long jxl = (long long)ix + dx, jyl = (long long)iy + dy;
      if (jxl < 0 || jyl < 0 || jxl >= side || jyl >= side) continue;
      const unsigned jx = (unsigned)jxl, jy = (unsigned)jyl;
      int j = b;
      if (dx != 0 || dy != 0) {
        const unsigned diff = (ix ^ jx) | (iy ^ jy);
        const int up = 32 - __clz(diff);  // levels to the common ancestor
        int a = b;
        for (int t = 0; t < up; ++t) a = iparent[a];
        for (int t = up - 1; t >= 0 && a >= 0; --t) {
          const int q = (int)((((jy >> t) & 1u) << 1) | ((jx >> t) & 1u));
          a = ichild[4 * a + q];
        }
        j = a;
      }
      if (j < 0) continue;
      // insertion by path code
      const unsigned long long cj = path_code(jx, jy);
      int k = cnt++;
      while (k > 0 && code[k - 1] > cj) {
        code[k] = code[k - 1];
        id[k] = id[k - 1];
        --k;
      }
      code[k] = cj;
      id[k] = j;
    }
  ncoll[i] = cnt;
  for (int k = 0; k < kMaxColl; ++k) coll[9 * i + k] = k < cnt ? id[k] : -1;
}

// *big = 1 if a leaf holds more than big_max sources or targets
__global__ void k_big_leaves(int64_t nb, const int* nchild, const int* ses, const int* set,
                             int big_max, int* big) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb || nchild[i] != 0) return;
  const int m = max(ses[2 * i + 1] - ses[2 * i], set[2 * i + 1] - set[2 * i]);
  if (m > big_max) *big = 1;
}

__global__ void k_root_coll(int* ncoll, int* coll) {
  ncoll[0] = 1;
  coll[0] = 0;
  for (int k = 1; k < 9; ++k) coll[k] = -1;
}

// ------------------------------------------------------------ level restriction
// flag pass (pts_tree2d.f:797-839): leaves among the grandparent's colleagues
// that touch the parent of a box at level lev.
// It only turns flags 0 into 1, so the levels (the reference sweeps them from
// the finest up) run in one launch; distest = 1.05 (bs_{l-1} + bs_{l-2}) / 2 of
// the box's level l comes from `dist`.
struct LevelReals {
  double v[kMaxLevels + 1];
};

__global__ void k_flag1(int64_t n, int lo, LevelReals dist, const int* ilevel, const int* iparent,
                        const int* ncoll, const int* coll, const int* nchild,
                        const double* centers, int* iflag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = lo + (int)i;
  const double distest = dist.v[ilevel[b]];
  const int dad = iparent[b];
  const int gd = iparent[dad];
  const double dx0 = centers[2 * dad], dy0 = centers[2 * dad + 1];
  for (int k = 0; k < ncoll[gd]; ++k) {
    const int j = coll[9 * gd + k];
    if (nchild[j] == 0 && iflag[j] == 0) {
      if (fabs(centers[2 * j] - dx0) <= distest && fabs(centers[2 * j + 1] - dy0) <= distest)
        iflag[j] = 1;
    }
  }
}

// flag+ pass (pts_tree2d.f:845-889): leaves among the parent's colleagues
// touching a flagged box.
__global__ void k_flag2(int64_t n, int lo, double distest, const int* iparent, const int* ncoll,
                        const int* coll, const int* nchild, const double* centers, int* iflag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = lo + (int)i;
  const int f = iflag[b];
  if (f != 1 && f != 2) return;
  const int dad = iparent[b];
  const double bx = centers[2 * b], by = centers[2 * b + 1];
  for (int k = 0; k < ncoll[dad]; ++k) {
    const int j = coll[9 * dad + k];
    if (nchild[j] == 0 && iflag[j] == 0) {
      if (fabs(centers[2 * j] - bx) <= distest && fabs(centers[2 * j + 1] - by) <= distest)
        iflag[j] = 2;
    }
  }
}

// ------------------------------------------------------------ reorganisation
// The new number of every box: the boxes are covered by segments (a level's
// original boxes, a level's tail boxes), sorted by first box; segment k moves
// [from[k], from[k+1]) to to[k], to[k] + 1, ...
constexpr int kMaxSeg = 2 * (kMaxLevels + 1);
struct SegTable {
  int n;
  int from[kMaxSeg], to[kMaxSeg];
};

__global__ void k_map_segments(int64_t nb, SegTable T, int* map) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb) return;
  int lo = 0, hi = T.n - 1;  // last segment with from <= i
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (T.from[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  map[i] = T.to[lo] + (int)(i - T.from[lo]);
}

__global__ void k_reorg_apply(int64_t n, const int* map, const double* c0, const int* lev0,
                              const int* par0, const int* nch0, const int* ich0, const int* fl0,
                              const int* s0, const int* t0, double* c1, int* lev1, int* par1,
                              int* nch1, int* ich1, int* fl1, int* s1, int* t1) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int m = map[i];
  c1[2 * m] = c0[2 * i];
  c1[2 * m + 1] = c0[2 * i + 1];
  lev1[m] = lev0[i];
  nch1[m] = nch0[i];
  fl1[m] = fl0[i] == 3 ? 3 : 0;  // the updateflags sweep starts from the flag-3 boxes
  s1[2 * m] = s0[2 * i];
  s1[2 * m + 1] = s0[2 * i + 1];
  t1[2 * m] = t0[2 * i];
  t1[2 * m + 1] = t0[2 * i + 1];
  par1[m] = par0[i] < 0 ? -1 : map[par0[i]];
  for (int q = 0; q < 4; ++q) ich1[4 * m + q] = ich0[4 * i + q] < 0 ? -1 : map[ich0[4 * i + q]];
}

// ------------------------------------------------------------ one-workgroup builds
// The refinement of trees and levels of a few thousand boxes is a chain of
// small dependent steps: as separate launches (flags, scan, next level,
// children; flags per level) each step costs a launch of ~2.4 us and the
// chain a host round trip of ~10 us per level, whatever its size.  One
// workgroup of 1024 threads runs the whole chain instead, with barriers
// between the steps.  Limits: kWgLevel boxes of a level in refinement (four
// per thread; beyond it the per-level launches spread over the CUs win) and
// kWgBoxes boxes in all in the flag passes (1765 boxes 5 us, 50000 250 us, where
// the launches take 60).
constexpr int kWgThreads = 1024;
constexpr int kWgWaves = kWgThreads / 64;
constexpr int kWgLevel = 4 * kWgThreads;
constexpr int kWgBoxes = 8192;

struct BoxPtrs {
  double* centers;
  int *ilevel, *iparent, *nchild, *ichild, *ncoll, *coll, *ses, *set, *iflag;
};

// State words of the kernels below: status, level, boxes, big-leaf flag
// (k_coll_walk), then two words per level.
constexpr int kStStatus = 0, kStLevel = 1, kStBoxes = 2, kStBig = 3, kStLev = 4;
constexpr int kStWords = kStLev + 2 * (kMaxLevels + 2);

// Level ranges and box sizes, by value
struct LevelTab {
  int ls[kMaxLevels + 1], le[kMaxLevels + 1];
  double bs[kMaxLevels + 1];
};

// digit_bounds3 by a whole wavefront: 21 probes per bound and round (a box of
// 1e6 points takes 5 rounds of dependent loads, not 20).
__device__ void digit_bounds3_wave(const Keys& K, int64_t lo0, int64_t hi0, int lev, int* b) {
  constexpr int kP = 21;
  const int lane = threadIdx.x & 63;
  const int q = min(lane / kP, 2), j = lane - q * kP;
  const bool in = lane < 3 * kP;
  int64_t lo = lo0, hi = hi0;
  while (__ballot(hi > lo)) {
    const int64_t w = hi - lo;
    const bool last = w <= kP;
    const int64_t pos = last ? lo + j : lo + (w * (j + 1)) / (kP + 1);
    const bool use = in && (last ? j < w : true) && w > 0;
    const bool below = use && digit_at(K, use ? pos : lo0, lev) < q + 1;
    const unsigned long long m = (__ballot(below) >> (q * kP)) & ((1ull << kP) - 1ull);
    const int c = __popcll(m);
    if (w > 0) {
      if (last) {
        lo = hi = lo + c;
      } else {
        const int64_t l1 = c > 0 ? lo + (w * c) / (kP + 1) + 1 : lo;
        const int64_t h1 = c < kP ? lo + (w * (c + 1)) / (kP + 1) : hi;
        lo = l1;
        hi = h1;
      }
    }
  }
  for (int k = 0; k < 3; ++k) b[k] = (int)__shfl(lo, k * kP, 64);
}

// the four children of box b by a whole wavefront (make_children_of, mode 0)
__device__ void make_children_wave(int b, int c0, double half, int lev, const BoxPtrs& B,
                                   const Keys& ks, const Keys& kt) {
  const int lane = threadIdx.x & 63;
  const int s0 = B.ses[2 * b], s1 = B.ses[2 * b + 1], t0 = B.set[2 * b], t1 = B.set[2 * b + 1];
  int bs[3], bt[3];
  digit_bounds3_wave(ks, s0, s1, lev, bs);
  digit_bounds3_wave(kt, t0, t1, lev, bt);
  if (lane < 4) {
    const int q = lane, c = c0 + q;
    B.centers[2 * c] = B.centers[2 * b] + ((q & 1) ? half : -half);
    B.centers[2 * c + 1] = B.centers[2 * b + 1] + ((q & 2) ? half : -half);
    B.iparent[c] = b;
    B.nchild[c] = 0;
    for (int k = 0; k < 4; ++k) B.ichild[4 * c + k] = -1;
    B.ichild[4 * b + q] = c;
    B.ilevel[c] = lev;
    B.ses[2 * c] = q == 0 ? s0 : q == 1 ? bs[0] : q == 2 ? bs[1] : bs[2];
    B.ses[2 * c + 1] = q == 0 ? bs[0] : q == 1 ? bs[1] : q == 2 ? bs[2] : s1;
    B.set[2 * c] = q == 0 ? t0 : q == 1 ? bt[0] : q == 2 ? bt[1] : bt[2];
    B.set[2 * c + 1] = q == 0 ? bt[0] : q == 1 ? bt[1] : q == 2 ? bt[2] : t1;
    B.iflag[c] = 0;
    if (q == 0) B.nchild[b] = 4;
  }
}

// Refinement (pts_tree2d.f:551-631) from level l0 on (0: from the root, made
// here) while levels hold at most kWgLevel boxes, keys reach (depth levels) and
// the boxes fit cap.  State: status 1 done (level = nlevels), 0 stopped before
// refining `level` (too many boxes, or keys too short), 2 the same for want of
// capacity; first box and count of every level made.
__global__ __launch_bounds__(kWgThreads) void k_refine_wg(const double* bounds, int ns, int nt,
                                                          int idivflag, int ndiv, int nlmax,
                                                          int depth, int cap, BoxPtrs B, Keys ks,
                                                          Keys kt, int l0, int* st) {
  __shared__ int list[kWgLevel];
  __shared__ int lds[kWgWaves + 1];
  const int tid = threadIdx.x, wave = tid >> 6;
  double cx0, cy0, bs0;
  root_square(bounds, &cx0, &cy0, &bs0);
  double h = 0.5 * bs0;
  for (int l = 0; l < l0; ++l) h *= 0.5;
  int lo = 0, n = 1, nb = 1;
  if (l0 == 0) {
    if (tid == 0) {
      B.centers[0] = cx0;
      B.centers[1] = cy0;
      B.ilevel[0] = 0;
      B.iparent[0] = -1;
      B.nchild[0] = 0;
      for (int q = 0; q < 4; ++q) B.ichild[q] = -1;
      B.ses[0] = 0;
      B.ses[1] = ns;
      B.set[0] = 0;
      B.set[1] = nt;
      B.iflag[0] = 0;
      st[kStBig] = 0;
      st[kStLev] = 0;
      st[kStLev + 1] = 1;
    }
  } else {
    nb = st[kStBoxes];
    lo = st[kStLev + 2 * l0];
    n = st[kStLev + 2 * l0 + 1];
  }
  __syncthreads();
  int l = l0, status = 0;
  for (;;) {
    if (l >= nlmax) {
      status = 1;
      break;
    }
    if (n > kWgLevel || l + 1 > depth) break;
    bool f[4];
    int c = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = 4 * tid + u;
      f[u] = i < n && box_full(lo + i, B.ses, B.set, idivflag, ndiv);
      c += f[u] ? 1 : 0;
    }
    int nref;
    int ex = block_exclusive_scan_w<kWgWaves>(c, lds, &nref);
    if (nref == 0) {
      status = 1;
      break;
    }
    if (nb + 4 * nref > cap) {
      status = 2;
      break;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (f[u]) list[ex++] = lo + 4 * tid + u;
    __syncthreads();
    h *= 0.5;
    if (nref <= 4 * kWgWaves) {
      for (int k = wave; k < nref; k += kWgWaves)
        make_children_wave(list[k], nb + 4 * k, h, l + 1, B, ks, kt);
    } else {
      for (int k = tid; k < nref; k += kWgThreads)
        make_children_of(list[k], nb + 4 * k, h, l + 1, B.centers, B.ilevel, B.iparent, B.nchild,
                         B.ichild, B.ses, B.set, B.iflag, 0, ks, kt);
    }
    __syncthreads();
    ++l;
    lo = nb;
    n = 4 * nref;
    nb += n;
    if (tid == 0) {
      st[kStLev + 2 * l] = lo;
      st[kStLev + 2 * l + 1] = n;
    }
  }
  if (tid == 0) {
    st[kStStatus] = status;
    st[kStLevel] = l;
    st[kStBoxes] = nb;
  }
}

// ------------------------------------------------------------ refinement from the keys
// The whole refinement at once where a box is refined for its sources alone
// (idivflag 0) and no refined box is as deep as the keys.  A box of level l is
// an interval of the sorted keys with common first l digits.  Let it start at
// source s; it holds more than ndiv sources exactly if the keys s and s + ndiv
// agree in l digits, and s starts a box of level l exactly if the keys s - 1
// and s do not.  So the refined boxes that start at s are those of the levels
//   common(s - 1, s) < l <= common(s, s + ndiv),
// known without the levels above.  In order of (level, s) they are the boxes
// that the level-by-level refinement refines, in its order (children are
// numbered by digit): the children of the refined box number p are 1 + 4 p ..
// 4 + 4 p, and its own number follows from its parent's place in the list.
//
// Four launches and one round trip for all levels: counts of every level per
// tile of keys, their prefix sums, the list, the boxes.  Level by level (one
// workgroup up to 4096 boxes a level, then two launches a level) it was a chain
// of up to 20 dependent steps: 0.52 ms at 1e6 points and 0.59 at 1e7, now 0.09
// and 0.32 (of which the boxes, with their binary searches, 0.06 and 0.19).
constexpr int kRkRows = kD1 + 1;  // levels 0 .. kD1 - 1, and the tiles that are too deep

__device__ __forceinline__ int common_digits(unsigned long long a, unsigned long long b, int d1) {
  const unsigned long long x = a ^ b;
  return x == 0 ? d1 : (__clzll((long long)x) - (64 - 2 * d1)) >> 1;
}

// A wavefront takes a tile of 64 * rounds keys.  EMIT 0: cnt[l][tile] = refined
// boxes of level l that start in the tile.  EMIT 1: their starts go to
// ref[levoff(l) + cnt[l][tile] (exclusive sums now) + rank].
template <int EMIT>
__global__ __launch_bounds__(256) void k_ref_keys(const unsigned long long* __restrict__ keys,
                                                  int ns, int ndiv, int d1, int nlmax, int rounds,
                                                  int ntiles, int* cnt, const int* tot, int refcap,
                                                  int* ref) {
  const int lane = threadIdx.x & 63, tile = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= ntiles) return;
  const int nl = min(d1, nlmax);  // levels that can be refined
  int c = 0;                      // lane l: counter of level l
  if (EMIT) {
    int v = lane < nl ? tot[lane] : 0;
    const int own = v;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
      const int u = __shfl_up(v, o, 64);
      if (lane >= o) v += u;
    }
    c = lane < nl ? v - own + cnt[(int64_t)lane * ntiles + tile] : 0;
  }
  const unsigned long long lt = (1ull << lane) - 1ull;
  bool deep = false;
  constexpr int U = 4;
  for (int r0 = 0; r0 < rounds; r0 += U) {
    unsigned long long k[U], kn[U], kp[U];
    const int64_t s0 = (int64_t)tile * 64 * rounds + (int64_t)r0 * 64 + lane;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = s0 + 64 * u;
      k[u] = keys[min(s, (int64_t)ns - 1)];
      kn[u] = keys[min(s + ndiv, (int64_t)ns - 1)];
      kp[u] = keys[min(max(s - 1, (int64_t)0), (int64_t)ns - 1)];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = s0 + 64 * u;
      const int cp = s > 0 ? common_digits(kp[u], k[u], d1) : -1;
      int w = s + ndiv < ns ? common_digits(k[u], kn[u], d1) : -1;
      if (w >= d1 && nlmax > d1) deep = true;
      w = min(w, nl - 1);
      const bool act = s < ns && w > cp;
      if (!__ballot(act)) continue;
      for (int l = 0; l < nl; ++l) {
        const bool mine = act && cp < l && l <= w;
        const unsigned long long m = __ballot(mine);
        if (!m) continue;
        if (EMIT) {
          const int at = __builtin_amdgcn_readlane(c, l) + __popcll(m & lt);
          if (mine && at < refcap) ref[at] = (int)s;
        }
        if (lane == l) c += __popcll(m);
      }
    }
  }
  if (!EMIT) {
    const bool any = __ballot(deep) != 0;
    if (lane < kD1) cnt[(int64_t)lane * ntiles + tile] = c;
    if (lane == kD1) cnt[(int64_t)lane * ntiles + tile] = any ? 1 : 0;
  }
}

// Exclusive sums of the rows of cnt, a workgroup a row; tot[row] its total.
__global__ __launch_bounds__(kScanThreads) void k_ref_scan(int ntiles, int* cnt, int* tot) {
  __shared__ int lds[kScanWaves + 1];
  int* row = cnt + (int64_t)blockIdx.x * ntiles;
  constexpr int U = 8;
  int carry = 0;
  for (int i0 = 0; i0 < ntiles; i0 += kScanThreads * U) {
    int v[U], s = 0, all;
    const int i = i0 + threadIdx.x * U;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = i + u < ntiles ? row[i + u] : 0;
      s += v[u];
    }
    int ex = carry + block_exclusive_scan(s, lds, &all);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i + u < ntiles) row[i + u] = ex;
      ex += v[u];
    }
    carry += all;
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

// first i in [lo, hi) with (k[i] >> sh) >= p, or hi
__device__ __forceinline__ int first_at_least(const unsigned long long* k, int lo, int hi, int sh,
                                              unsigned long long p) {
  while (lo < hi) {
    const int mid = lo + ((hi - lo) >> 1);
    if ((k[mid] >> sh) < p) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// The boxes: a thread writes the four children of a refined box (nchild of a
// child from its count, ichild of a child only if it is a leaf).  Block 0 writes
// the state: status 1 done, 2 more than cap boxes, 3 deeper than the keys.
__global__ __launch_bounds__(256) void k_ref_make(const double* bounds, int ns, int nt, int ndiv,
                                                  int nlmax, int cap, const int* tot,
                                                  const int* ref, BoxPtrs B, Keys ks, Keys kt,
                                                  int* st) {
  __shared__ int off[kD1 + 2];
  const int d1 = ks.d1, nl = min(d1, nlmax);
  if (threadIdx.x == 0) {
    off[0] = 0;
    for (int l = 0; l < nl; ++l) off[l + 1] = off[l] + tot[l];
  }
  __syncthreads();
  const int R = off[nl];
  const int status = tot[kD1] > 0 ? 3 : 1 + 4 * (int64_t)R > cap ? 2 : 1;
  double cx0, cy0, bs0;
  root_square(bounds, &cx0, &cy0, &bs0);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    int top = 0;
    while (top < nl && tot[top] > 0) ++top;
    st[kStStatus] = status;
    st[kStLevel] = top;
    st[kStBoxes] = 1 + 4 * R;
    st[kStBig] = 0;
    st[kStLev] = 0;
    st[kStLev + 1] = 1;
    for (int l = 1; l <= top; ++l) {
      st[kStLev + 2 * l] = 1 + 4 * off[l - 1];
      st[kStLev + 2 * l + 1] = 4 * tot[l - 1];
    }
    if (status == 1) {
      B.centers[0] = cx0;
      B.centers[1] = cy0;
      B.ilevel[0] = 0;
      B.iparent[0] = -1;
      B.nchild[0] = R > 0 ? 4 : 0;
      if (R == 0)
        for (int q = 0; q < 4; ++q) B.ichild[q] = -1;
      B.ses[0] = 0;
      B.ses[1] = ns;
      B.set[0] = 0;
      B.set[1] = nt;
      B.iflag[0] = 0;
    }
  }
  if (status != 1) return;
  for (int p = blockIdx.x * 256 + threadIdx.x; p < R; p += gridDim.x * 256) {
    int l = 0;
    while (off[l + 1] <= p) ++l;
    const int s = ref[p];
    const unsigned long long key = ks.k1[s];
    // its own number: the last refined box of level l - 1 that starts at or before s
    int own = 0;
    if (l > 0) {
      int lo = off[l - 1], hi = off[l] - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (ref[mid] <= s) lo = mid;
        else hi = mid - 1;
      }
      own = 1 + 4 * lo + (int)((key >> (2 * (d1 - l))) & 3ull);
    }
    // its end: keys s .. s + ndiv are inside; doubling steps, then bisection
    const int sh = 2 * (d1 - l);
    const unsigned long long P = key >> sh;
    int in = s + ndiv, end = ns;
    int64_t step = (int64_t)ndiv + 1;
    if (l > 0) {
      for (;;) {
        if (step >= ns - in) break;  // (else in + step < ns)
        if ((ks.k1[in + step] >> sh) != P) {
          end = in + (int)step;
          break;
        }
        in += (int)step;
        step *= 2;
      }
      end = first_at_least(ks.k1, in + 1, end, sh, P + 1);
    }
    int t0 = 0, t1 = nt;
    if (l > 0 && nt > 0) {
      t0 = first_at_least(kt.k1, 0, nt, sh, P);
      t1 = first_at_least(kt.k1, t0, nt, sh, P + 1);
    }
    int bs[5] = {s, 0, 0, 0, end}, bt[5] = {t0, t0, t0, t0, t1};
    int64_t bq[3];
    digit_bounds3(ks, s, end, l + 1, bq);
    for (int q = 1; q < 4; ++q) bs[q] = (int)bq[q - 1];
    digit_bounds3(kt, t0, t1, l + 1, bq);
    for (int q = 1; q < 4; ++q) bt[q] = (int)bq[q - 1];
    // its centre, by the centre arithmetic of path_key
    double cx = cx0, cy = cy0, h = 0.5 * bs0;
    for (int k = 1; k <= l; ++k) {
      const int g = (int)(key >> (2 * (d1 - k))) & 3;
      h *= 0.5;
      cx += (g & 1) ? h : -h;
      cy += (g & 2) ? h : -h;
    }
    h *= 0.5;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 1 + 4 * p + q;
      const bool full = bs[q + 1] - bs[q] > ndiv && l + 1 < nlmax;
      B.centers[2 * c] = cx + ((q & 1) ? h : -h);
      B.centers[2 * c + 1] = cy + ((q & 2) ? h : -h);
      B.iparent[c] = own;
      B.nchild[c] = full ? 4 : 0;
      if (!full)
        for (int k = 0; k < 4; ++k) B.ichild[4 * c + k] = -1;
      B.ichild[4 * own + q] = c;
      B.ilevel[c] = l + 1;
      B.ses[2 * c] = bs[q];
      B.ses[2 * c + 1] = bs[q + 1];
      B.set[2 * c] = bt[q];
      B.set[2 * c + 1] = bt[q + 1];
      B.iflag[c] = 0;
    }
  }
}

// The flag+ passes (k_flag2, finest level first) and the refinement of every
// flagged box of levels 1 .. nl-2 (refine_segments over the levels in order).
// State: boxes; per level the first and last of its new boxes; status 1: cap
// boxes are too few (5 nb never are, each box is refined at most once), and the
// kernel has to run again with more, which repeats what it has done.
__global__ __launch_bounds__(kWgThreads) void k_flags_wg(LevelTab T, int nl, int nb, int cap,
                                                         BoxPtrs B, Keys ks, Keys kt, int* st) {
  __shared__ int list[kWgLevel];
  __shared__ int lds[kWgWaves + 1];
  __shared__ int cnt, per[kMaxLevels + 2];
  const int tid = threadIdx.x;
  for (int k = tid; k < kMaxLevels + 2; k += kWgThreads) per[k] = 0;
  for (int l = nl; l >= 1; --l) {
    const double distest = 1.05 * (T.bs[l] + T.bs[l - 1]) / 2.0;
    const int lo = T.ls[l], n = T.le[l] - lo;
    for (int r0 = 0; r0 < n; r0 += kWgLevel) {
      if (tid == 0) cnt = 0;
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = r0 + u * kWgThreads + tid;
        const int f = i < n ? B.iflag[lo + i] : 0;
        if (f == 1 || f == 2) list[atomicAdd(&cnt, 1)] = lo + i;
      }
      __syncthreads();
      const int m = cnt;
      for (int t = tid; t < 16 * m; t += kWgThreads) {
        const int b = list[t >> 4], k = t & 15;
        const int dad = B.iparent[b];
        if (k >= B.ncoll[dad]) continue;
        const int j = B.coll[9 * dad + k];
        if (B.nchild[j] == 0 && B.iflag[j] == 0 &&
            fabs(B.centers[2 * j] - B.centers[2 * b]) <= distest &&
            fabs(B.centers[2 * j + 1] - B.centers[2 * b + 1]) <= distest)
          B.iflag[j] = 2;
      }
      __syncthreads();
    }
  }
  const int nb0 = nb;
  int status = 0;
  if (nl >= 3) {
    const int lo = T.ls[1], n = T.le[nl - 2] - lo;
    for (int r0 = 0; r0 < n; r0 += kWgLevel) {
      bool f[4];
      int c = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = r0 + 4 * tid + u;
        f[u] = i < n && B.iflag[lo + i] > 0;
        c += f[u] ? 1 : 0;
      }
      int nref;
      int ex = block_exclusive_scan_w<kWgWaves>(c, lds, &nref);
      if (nref == 0) continue;  // uniform
      if (nb + 4 * nref > cap) {
        status = 1;
        break;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (f[u]) list[ex++] = lo + r0 + 4 * tid + u;
      __syncthreads();
      for (int k = tid; k < nref; k += kWgThreads) {
        const int b = list[k], lev = B.ilevel[b] + 1;
        atomicAdd(&per[lev], 1);
        make_children_of(b, nb + 4 * k, 0.5 * T.bs[lev], lev, B.centers, B.ilevel, B.iparent,
                         B.nchild, B.ichild, B.ses, B.set, B.iflag, 1, ks, kt);
      }
      nb += 4 * nref;
      __syncthreads();
    }
  }
  __syncthreads();
  if (tid == 0) {
    int at = nb0;
    for (int l = 0; l <= nl; ++l) {
      st[kStLev + 2 * l] = at;
      at += 4 * per[l];
      st[kStLev + 2 * l + 1] = at;
    }
    st[kStStatus] = status;
    st[kStBoxes] = nb;
  }
}

// ------------------------------------------------------------ restriction sweeps
// A sweep's boxes: n1 boxes from lo1 on, then the tail boxes [ts, te) of the
// state words.  kLrTile boxes a workgroup of 256 threads, 16 lanes a box where
// a box looks at its (parent's) colleagues.  Capacity and launch bounds of the
// updateflags sweep are guesses (cap, tail_ub); a level that would pass them sets
// the status word and makes nothing, and the caller builds again with more room.
constexpr int kLrTile = 64;

struct LrSeq {
  int n1, lo1, ts, te;
  __device__ int n() const { return n1 + (te - ts); }
  __device__ int box(int i) const { return i < n1 ? lo1 + i : ts + (i - n1); }
};

// flagged boxes (iflag > 0) of every kLrTile of the n boxes from lo on, and, by
// the level of their children, in the state words (zero before)
__global__ __launch_bounds__(256) void k_flag_count(int n, int lo, const int* iflag,
                                                    const int* ilevel, int* part, int* st) {
  __shared__ int per[kMaxLevels + 2];
  for (int k = threadIdx.x; k < kMaxLevels + 2; k += 256) per[k] = 0;
  __syncthreads();
  const int i = blockIdx.x * 256 + threadIdx.x;
  const bool f = i < n && iflag[lo + i] > 0;
  const unsigned long long m = __ballot(f);
  if ((threadIdx.x & 63) == 0 && i < n) part[i / kLrTile] = __popcll(m);
  if (f) atomicAdd(&per[ilevel[lo + i] + 1], 1);
  __syncthreads();
  for (int k = threadIdx.x; k < kMaxLevels + 2; k += 256)
    if (per[k]) atomicAdd(&st[kStLev + 2 * k], per[k]);
}

// Children of the flagged boxes of a sweep, numbered in sweep order from nb on
// (make_children_of, mode 1).  SWEEP: level l of the updateflags sweep, nb = te
// of that level, the new range is level l+1's; else the levels 1 .. nl-2 at
// once, which k_flag_count has counted.
template <int SWEEP>
__global__ __launch_bounds__(256) void k_flag_children(int n1, int lo1, int l, int nb,
                                                       const int* part, LevelTab T, int cap,
                                                       BoxPtrs B, Keys ks, Keys kt, int* st) {
  __shared__ int lds[kScanWaves + 1];
  LrSeq q{n1, lo1, 0, 0};
  if (SWEEP) {
    q.ts = st[kStLev + 2 * l];
    q.te = nb = st[kStLev + 2 * l + 1];
  }
  const int n = q.n(), i0 = blockIdx.x * 256, i = i0 + threadIdx.x;
  if (i0 >= n && blockIdx.x > 0) return;
  const int b = i < n ? q.box(i) : 0;
  const bool f = i < n && B.iflag[b] > 0;
  const int carry = sum_parts(part, min(i0, n) / kLrTile, lds);
  int own;
  const int ex = block_exclusive_scan(f ? 1 : 0, lds, &own);
  const bool fits = nb + 4 * (int64_t)(carry + own) <= cap;
  if (!fits && threadIdx.x == 0) st[kStStatus] = 1;
  if (SWEEP && i0 + 256 >= n && threadIdx.x == 0) {
    st[kStLev + 2 * (l + 1)] = nb;
    st[kStLev + 2 * (l + 1) + 1] = fits ? nb + 4 * (carry + own) : nb;
  }
  if (f && fits) {
    const int lev = SWEEP ? l + 1 : B.ilevel[b] + 1;
    make_children_of(b, nb + 4 * (carry + ex), 0.5 * T.bs[lev], lev, B.centers, B.ilevel,
                     B.iparent, B.nchild, B.ichild, B.ses, B.set, B.iflag, 1, ks, kt);
  }
}

// Level l of the updateflags sweep (tree_routs2d.f:217-326, pts_tree2d.f:
// 940-1010): the tail boxes get their colleagues (k_coll's entries, in
// (parent's colleague, child slot) order), then the flag-3 boxes keep their
// flag, as 1, where a child of a colleague is refined and touches them.
__global__ __launch_bounds__(256) void k_sweep_flags(int n1, int lo1, int l, int tail_ub,
                                                     double lim, double distest, BoxPtrs B,
                                                     int* part, int* st) {
  __shared__ int list[kLrTile], hit[kLrTile];
  __shared__ int cnt;
  const LrSeq q{n1, lo1, st[kStLev + 2 * l], st[kStLev + 2 * l + 1]};
  const int n = q.n(), i0 = blockIdx.x * kLrTile;
  if (i0 >= n) return;
  const int tid = threadIdx.x, lane = tid & 63;
  if (blockIdx.x == 0 && tid == 0 && q.te - q.ts > tail_ub) st[kStStatus] = 1;
  if (i0 + kLrTile > n1) {
    for (int r = 0; r < kLrTile; r += 16) {
      const int i = i0 + r + (tid >> 4), k = lane & 15;
      const bool act = i >= n1 && i < n;
      const int b = act ? q.box(i) : 0;
      const int dad = act ? B.iparent[b] : 0;
      const double bx = B.centers[2 * b], by = B.centers[2 * b + 1];
      int id[4] = {-1, -1, -1, -1};
      if (act && k < B.ncoll[dad]) {
        const int j = B.coll[9 * dad + k];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int kb = B.ichild[4 * j + c];
          if (kb >= 0 && fabs(B.centers[2 * kb] - bx) <= lim &&
              fabs(B.centers[2 * kb + 1] - by) <= lim)
            id[c] = kb;
        }
      }
      const unsigned long long seg = 0xffffull << (lane & 48), lt = (1ull << lane) - 1ull;
      int at = 0, tot = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const unsigned long long m = __ballot(id[c] >= 0) & seg;
        at += __popcll(m & lt);
        tot += __popcll(m);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (id[c] >= 0) {
          if (at < kMaxColl) B.coll[9 * b + at] = id[c];
          ++at;
        }
      tot = min(tot, kMaxColl);
      if (act && k == 0) B.ncoll[b] = tot;
      if (act && k >= tot && k < kMaxColl) B.coll[9 * b + k] = -1;
    }
  }
  if (tid < kLrTile) {  // the first wavefront
    const int i = i0 + tid;
    const int b = i < n ? q.box(i) : 0;
    const bool f = i < n && B.iflag[b] == 3;
    const unsigned long long m = __ballot(f);
    const int at = __popcll(m & ((1ull << tid) - 1ull));
    if (f) list[at] = b;
    hit[tid] = 0;
    if (tid == 0) cnt = __popcll(m);
  }
  __syncthreads();  // (the colleagues above are visible to the workgroup too)
  const int m = cnt;
  for (int t = tid; t < 16 * m; t += 256) {
    const int b = list[t >> 4], k = t & 15;
    if (k >= B.ncoll[b]) continue;
    const int j = B.coll[9 * b + k];
    const double bx = B.centers[2 * b], by = B.centers[2 * b + 1];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int kb = B.ichild[4 * j + c];
      any = any || (kb >= 0 && B.nchild[kb] > 0 && fabs(B.centers[2 * kb] - bx) <= distest &&
                    fabs(B.centers[2 * kb + 1] - by) <= distest);
    }
    if (any) hit[t >> 4] = 1;
  }
  __syncthreads();
  if (tid < kLrTile) {
    const bool h = tid < m && hit[tid] != 0;
    if (tid < m) B.iflag[list[tid]] = h ? 1 : 0;
    const unsigned long long k = __ballot(h);
    if (tid == 0) part[blockIdx.x] = __popcll(k);
  }
}

// ------------------------------------------------------------ final point order
// Positions in path order are the reference's point positions up to the order
// inside each leaf, which the reference keeps in input order: label every
// point (in input order) with its leaf's first position, then stable-sort.
__global__ void k_leaf_label(int64_t n, const int* nchild, const int* se, const int* perm,
                             unsigned long long* label) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n || nchild[b] != 0) return;
  const int s = se[2 * b];
  for (int i = s; i < se[2 * b + 1]; ++i) label[perm[i]] = (unsigned long long)s;
}

// The same order without the sort: inside each leaf (a contiguous range of
// the path order) the input indices in increasing order, placed by rank, one
// thread per point (leaves of up to kLeafRankMax points).  blockIdx.y: sources,
// targets.
constexpr int kLeafRankMax = 2048;

struct LeafOrder {
  int64_t n[2];
  const int* leaf[2];
  const int* se[2];
  const int* perm[2];
  int* out[2];
};

__global__ __launch_bounds__(256) void k_leaf_rank(LeafOrder a) {
  const int y = blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n[y]) return;
  const int b = a.leaf[y][i];
  const int s = a.se[y][2 * (int64_t)b], e = a.se[y][2 * (int64_t)b + 1];
  const int* p = a.perm[y];
  const int v = p[i];
  int rank = 0;
  int j = s;
  for (; j + 4 <= e; j += 4) {
    const int q0 = p[j], q1 = p[j + 1], q2 = p[j + 2], q3 = p[j + 3];
    rank += (q0 < v) + (q1 < v) + (q2 < v) + (q3 < v);
  }
  for (; j < e; ++j) rank += p[j] < v ? 1 : 0;
  a.out[y][s + rank] = v;
}

// leaf[i] = the leaf holding sorted point i, for sources and targets
// (blockIdx.y).  A wavefront takes 64 boxes and writes their point ranges one
// box after the other with all 64 lanes (consecutive lanes on consecutive
// points).
__global__ void k_leaf_of(int64_t n, const int* nchild, const int* ses, const int* set,
                          int* leaf_s, int* leaf_t) {
  const int* se = blockIdx.y ? set : ses;
  int* leaf = blockIdx.y ? leaf_t : leaf_s;
  const int lane = threadIdx.x & 63;
  const int64_t b0 = (int64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63);
  const int64_t b = b0 + lane;
  int s = 0, e = 0;
  if (b < n && nchild[b] == 0) {
    s = se[2 * b];
    e = se[2 * b + 1];
  }
  for (int k = 0; k < 64; ++k) {
    const int sk = __builtin_amdgcn_readlane(s, k), ek = __builtin_amdgcn_readlane(e, k);
    for (int i = sk + lane; i < ek; i += 64) leaf[i] = (int)(b0 + k);
  }
}

// ------------------------------------------------------------ host helpers
// Points of one set (sources or targets) sorted by path key.
struct PathKeys {
  int64_t n = 0;
  int d1 = 0, d2 = 0;
  DBuf<unsigned long long> k1, k2;  // sorted
  DBuf<int> perm;                   // sorted position -> input index
  Keys view() const { return Keys{k1.p, k2.p, d1, d2}; }

  void alloc(int64_t np, int dd1, int dd2, hipStream_t st) {
    n = np;
    d1 = dd1;
    d2 = dd2;
    perm.alloc(std::max<int64_t>(n, 1), st);
    k1.alloc(std::max<int64_t>(n, 1), st);
    k2.alloc(d2 > 0 ? std::max<int64_t>(n, 1) : 0, st);
  }
  // keys of both words (deep trees)
  void build(const double* xy, int64_t np, double cx, double cy, double bs, int dd1, int dd2,
             hipStream_t st) {
    alloc(np, dd1, dd2, st);
    if (n == 0) return;
    DBuf<unsigned long long> u1(n, st), u2(n, st);
    launch1d(k_path_keys, n, st, xy, cx, cy, bs, d1, d2, u1.p, u2.p);
    // lexicographic (key1, key2): stable LSD passes, key2 first
    DBuf<unsigned long long> t2(n, st), t1(n, st);
    DBuf<int> p1(n, st);
    radix_sort(u2.p, t2.p, nullptr, p1.p, n, 2 * d2, st);
    launch1d(k_gather_by<unsigned long long>, n, st, p1.p, u1.p, t1.p);
    radix_sort(t1.p, k1.p, p1.p, perm.p, n, 2 * d1, st);
    launch1d(k_gather_by<unsigned long long>, n, st, perm.p, u2.p, k2.p);
  }
};

inline BoxPtrs ptrs(const Boxes& b) {
  return BoxPtrs{b.centers.p, b.ilevel.p, b.iparent.p, b.nchild.p, b.ichild.p,
                 b.ncoll.p,   b.coll.p,   b.ses.p,     b.set.p,    b.iflag.p};
}

struct Builder {
  hipStream_t st;
  Boxes B;
  int nboxes = 0;
  DBuf<int> flag, offs, total;
  Keys ks{}, kt{};
  // the centre comparisons of k_coll_walk are exact when the domain is not far
  // from the origin relative to its size
  bool walk_ok = false;

  explicit Builder(hipStream_t s) : st(s) { total.alloc(64, s); }

  void scan_only(int n) { exclusive_scan(flag.p, offs.p, n, (int*)nullptr, st); }
  // exclusive scan of flag[0..n) into offs, returns the total
  int scan(int n) {
    if (n <= 0) return 0;
    scan_only(n);
    hipLaunchKernelGGL(k_total, dim3(1), dim3(1), 0, st, n, flag.p, offs.p, total.p);
    int h = 0;
    readback(&h, total.p, sizeof(int), st);
    return h;
  }
  void ensure_flag(int n) {
    if ((size_t)n > flag.n) {
      flag.alloc(std::max<size_t>(n, 2 * flag.n), st);
      offs.alloc(flag.n, st);
    }
  }
  // refine the boxes lo..lo+n-1 selected by flag[]; returns the count refined
  int refine(int lo, int n, double bs_child, int lev, int mode) {
    const int nref = scan(n);
    if (nref == 0) return 0;
    B.grow(nboxes + 4 * (size_t)nref, nboxes);
    launch1d(k_make_children, n, st, lo, flag.p, offs.p, nboxes, 0.5 * bs_child, lev,
             B.centers.p, B.ilevel.p, B.iparent.p, B.nchild.p, B.ichild.p, B.ses.p, B.set.p,
             B.iflag.p, mode, ks, kt);
    nboxes += 4 * nref;
    return nref;
  }
  void computecoll(const std::vector<int>& ls, const std::vector<int>& le,
                   const std::vector<double>& bs, int nlevels, int* big = nullptr) {
    B.alloc_coll(nboxes);
    // all levels at once by walking the tree from every box (integer
    // coordinates exact: at most kWalkLevels levels, domain near the origin)
    if (nlevels <= kWalkLevels && walk_ok) {
      launch1d(k_coll_walk, nboxes, st, B.ilevel.p, B.iparent.p, B.ichild.p, B.centers.p,
               B.ncoll.p, B.coll.p, B.nchild.p, B.ses.p, B.set.p, kLeafRankMax, big);
      return;
    }
    if (big)
      launch1d(k_big_leaves, nboxes, st, B.nchild.p, B.ses.p, B.set.p, kLeafRankMax, big);
    hipLaunchKernelGGL(k_root_coll, dim3(1), dim3(1), 0, st, B.ncoll.p, B.coll.p);
    for (int l = 1; l <= nlevels; ++l)
      launch1d(k_coll, le[l] - ls[l], st, ls[l], bs[l], B.iparent.p, B.ichild.p, B.centers.p,
               B.ncoll.p, B.coll.p);
  }
  // pts_tree_reorg: per level >= 2, original boxes then the tail boxes; the
  // arrays then have room for cap boxes.
  void reorg(std::vector<int>& ls, std::vector<int>& le, const std::vector<int>& ts,
             const std::vector<int>& te, int nlevels, size_t cap) {
    DBuf<int> map(nboxes, st);
    std::vector<std::pair<int, int>> seg;  // (from, to) of non-empty segments
    for (int l = 0; l <= std::min(1, nlevels); ++l)
      if (le[l] > ls[l]) seg.push_back({ls[l], ls[l]});
    int cur = (nlevels >= 2) ? ls[2] : 0;
    for (int l = 2; l <= nlevels; ++l) {
      const int s = cur;
      if (le[l] > ls[l]) seg.push_back({ls[l], cur});
      cur += le[l] - ls[l];
      if (te[l] > ts[l]) seg.push_back({ts[l], cur});
      cur += te[l] - ts[l];
      ls[l] = s;
      le[l] = cur;
    }
    std::sort(seg.begin(), seg.end());
    SegTable T{};
    T.n = (int)seg.size();
    if (T.n > kMaxSeg) throw HipError{hipErrorInvalidValue, "tree reorganisation segments"};
    for (int k = 0; k < T.n; ++k) {
      T.from[k] = seg[k].first;
      T.to[k] = seg[k].second;
    }
    launch1d(k_map_segments, nboxes, st, T, map.p);
    Boxes N;
    N.alloc(cap, st);
    launch1d(k_reorg_apply, nboxes, st, map.p, B.centers.p, B.ilevel.p, B.iparent.p, B.nchild.p,
             B.ichild.p, B.iflag.p, B.ses.p, B.set.p, N.centers.p, N.ilevel.p, N.iparent.p,
             N.nchild.p, N.ichild.p, N.iflag.p, N.ses.p, N.set.p);
    B.swap_boxes(N);
  }
};

}  // namespace

// The steps of the tree build that do not depend on the leaf capacity: the
// bounding square, the box sizes, the points' path keys sorted (sources and
// targets separately).  Kept by a caller that needs the sorted keys before it
// chooses the leaf capacity (the parameter proposer) and handed to the build.
struct TreePrep {
  const double* src = nullptr;
  const double* trg = nullptr;
  int64_t ns = 0, nt = 0;
  int nlmax = 0;
  std::vector<double> bsall;  // box size of every possible level
  double root[2] = {0.0, 0.0};
  bool walk_ok = false;
  DBuf<double> bounds;        // min x, max x, min y, max y on the device
  PathKeys pk[2];
};

namespace {
void prepare_into(TreePrep& P, const double* src, int64_t ns, const double* trg, int64_t nt,
                  int nlmax, hipStream_t st) {
  if (nlmax > kMaxLevels) throw HipError{hipErrorInvalidValue, "nlmax beyond 51"};
  P.src = src;
  P.trg = trg;
  P.ns = ns;
  P.nt = nt;
  P.nlmax = nlmax;
  const int d1 = std::min(kD1, nlmax);
  P.pk[0].alloc(ns, d1, 0, st);
  P.pk[1].alloc(nt, d1, 0, st);
  P.bounds.alloc(4, st);
  // bounds, keys with their digit counts, one launch per digit
  const int nb = (int)std::min<int64_t>(kRedBlocks, std::max<int64_t>(1, ceil_div(ns + nt, 256)));
  DBuf<double> part(4 * nb, st);
  DBuf<unsigned long long> u0(ns, st), u1(nt, st);
  RsPlan rs;
  rs.init(ns, nt, 2 * d1, st);
  hipLaunchKernelGGL(k_bbox_partial, dim3(nb), dim3(256), 0, st, src, ns, trg, nt, part.p,
                     rs.words.p, (int64_t)rs.words.n);
  const int64_t m = std::max(ns, nt);
  hipLaunchKernelGGL(k_keys_count,
                     dim3(rs_count_grid(m), nt > 0 ? 2 : 1), dim3(kRsCountThreads), 0, st, src, ns, trg, nt, (const double*)part.p, nb, d1, rs.npass,
                     u0.p, u1.p, rs.hist(0), P.bounds.p);
  hip_throw(hipGetLastError(), "path keys");
  const unsigned long long* ki[2] = {u0.p, u1.p};
  unsigned long long* ko[2] = {P.pk[0].k1.p, P.pk[1].k1.p};
  int* vo[2] = {P.pk[0].perm.p, P.pk[1].perm.p};
  rs.sort(ki, ko, nullptr, vo, st);
}

// the host's share of a preparation, from the bounds
void prepare_host(TreePrep& P, const double* bb) {
  double bs0;
  root_square(bb, &P.root[0], &P.root[1], &bs0);
  // box sizes of every possible level (boxsize(l+1) = boxsize(l)/2)
  P.bsall.assign(P.nlmax + 2, 0.0);
  P.bsall[0] = bs0;
  for (int l = 1; l < (int)P.bsall.size(); ++l) P.bsall[l] = P.bsall[l - 1] / 2;
  P.walk_ok = std::max(std::fabs(P.root[0]), std::fabs(P.root[1])) <= std::ldexp(bs0, 20);
}
}  // namespace

TreePrep* tree_prepare(const double* src, int64_t ns, const double* trg, int64_t nt, int nlmax,
                       hipStream_t st) {
  std::unique_ptr<TreePrep> P(new TreePrep());
  prepare_into(*P, src, ns, trg, nt, nlmax, st);
  double bb[4];
  readback(bb, P->bounds.p, sizeof(bb), st);
  prepare_host(*P, bb);
  return P.release();
}

void tree_prepare_free(TreePrep* p) { delete p; }

bool tree_prepare_matches(const TreePrep* p, const double* src, int64_t ns, const double* trg,
                          int64_t nt, int nlmax) {
  return p && p->src == src && p->ns == ns && p->nt == nt && (nt == 0 || p->trg == trg) &&
         p->nlmax == nlmax;
}

// One build with `room` times the usual reserve for the boxes that the
// updateflags sweep adds (false: it needs more).
static bool build_try(const TreePrep* P, TreePrep* own, const double* src, int64_t ns,
                      const double* trg, int64_t nt, int ndiv, int idivflag, int nlmax, Tree& t,
                      hipStream_t st, int room) {
  Builder bld(st);
  t.ns = ns;
  t.nt = nt;
  const int d1 = std::min(kD1, nlmax);
  // the keys in use: the prepared ones, or deeper ones made below (points
  // closer than 2^-21 of the domain)
  PathKeys pkx[2];
  const PathKeys* pk[2] = {&P->pk[0], &P->pk[1]};
  bld.ks = pk[0]->view();
  bld.kt = pk[1]->view();

  // the refinement makes 2 to 3 boxes for every ndiv points of an area, 5 on a
  // curve, and the level restriction as many again on a curve, twice as many
  // around a few clusters, for which small trees, whose restriction would run
  // again, have room
  const size_t boxes = (size_t)((ns + nt) / std::max(ndiv, 1));
  bld.B.alloc(std::max<size_t>(2048, boxes <= kWgBoxes / 4 ? 18 * boxes : 11 * boxes), st);
  DBuf<int> state(kStWords, st);
  std::vector<int> hs(kStWords, 0);

  // ---- level-by-level refinement (pts_tree2d.f:551-631): by one workgroup
  // while the levels are small, else in batches.  While the bound on a level's
  // size is moderate, kBatch levels run between host synchronisations (level
  // ranges kept on the device); a refined box holds more than ndiv points, so
  // a level has at most 4 (ns + nt) / (ndiv + 1) boxes.  Otherwise, and for the
  // key-extension check at level d1, one level at a time with its exact count.
  auto refine_wg = [&](int l0) {
    hipLaunchKernelGGL(k_refine_wg, dim3(1), dim3(kWgThreads), 0, st,
                       (const double*)P->bounds.p, (int)ns, (int)nt, idivflag, ndiv, nlmax,
                       pk[0]->d1 + pk[0]->d2, (int)std::min<size_t>(bld.B.cap, INT32_MAX),
                       ptrs(bld.B), bld.ks, bld.kt, l0, state.p);
    hip_throw(hipGetLastError(), "refine");
  };
  // ... or from the keys, all levels at once
  const bool by_keys = idivflag == 0 && ndiv >= 1 && ns > 0 && nlmax >= 1;
  const int rounds = ns <= (1 << 20) ? 4 : 16;
  const int ntiles = by_keys ? (int)ceil_div(ns, 64 * rounds) : 0;
  DBuf<int> kcnt((size_t)kRkRows * ntiles, st), ktot(kRkRows, st), kref;
  auto refine_keys = [&](bool count) {
    const int cap = (int)std::min<size_t>(bld.B.cap, INT32_MAX);
    const unsigned long long* k = pk[0]->k1.p;
    const dim3 grid((ntiles + 3) / 4), blk(256);
    if (count) {
      hipLaunchKernelGGL(k_ref_keys<0>, grid, blk, 0, st, k, (int)ns, ndiv, pk[0]->d1, nlmax,
                         rounds, ntiles, kcnt.p, (const int*)nullptr, 0, (int*)nullptr);
      hipLaunchKernelGGL(k_ref_scan, dim3(kRkRows), dim3(kScanThreads), 0, st, ntiles, kcnt.p,
                         ktot.p);
    }
    kref.alloc(cap / 4 + 1, st);
    hipLaunchKernelGGL(k_ref_keys<1>, grid, blk, 0, st, k, (int)ns, ndiv, pk[0]->d1, nlmax,
                       rounds, ntiles, kcnt.p, (const int*)ktot.p, cap / 4 + 1, kref.p);
    hipLaunchKernelGGL(k_ref_make, dim3(std::min(ceil_div(cap / 4 + 1, 256), 2048u)), blk, 0, st,
                       (const double*)P->bounds.p, (int)ns, (int)nt, ndiv, nlmax, cap,
                       (const int*)ktot.p, (const int*)kref.p, ptrs(bld.B), bld.ks, bld.kt,
                       state.p);
    hip_throw(hipGetLastError(), "refine");
  };
  if (by_keys) refine_keys(true);
  else refine_wg(0);
  if (own && own->bsall.empty()) {
    // the bounds with the state, in one round trip
    double bb[4];
    readback2(hs.data(), state.p, sizeof(int) * kStWords, bb, own->bounds.p, sizeof(bb), st);
    prepare_host(*own, bb);
  } else {
    readback(hs.data(), state.p, sizeof(int) * kStWords, st);
  }
  if (by_keys && hs[kStStatus] == 2) {  // more boxes than expected
    bld.B.fit((size_t)hs[kStBoxes] + 64, 0);
    refine_keys(false);
    hs[kStStatus] = 1;
  } else if (by_keys && hs[kStStatus] == 3) {
    refine_wg(0);
    readback(hs.data(), state.p, sizeof(int) * kStWords, st);
  }
  kref.reset();
  kcnt.reset();
  const std::vector<double>& bsall = P->bsall;
  const double* root = P->root;
  bld.walk_ok = P->walk_ok;
  std::vector<int> ls{0}, le{1};
  std::vector<double> bs{bsall[0]};
  int nlevels = nlmax;
  const int64_t lev_cap = 4 * ((ns + nt) / (std::max(ndiv, 0) + 1) + 1);
  DBuf<int> dlev(2 * (nlmax + 2), st);
  int l = 0;
  bool done = false;
  // the levels that a one-workgroup run added
  auto take_wg = [&]() {
    bld.nboxes = hs[kStBoxes];
    for (int k = l + 1; k <= hs[kStLevel]; ++k) {
      bs.push_back(bsall[k]);
      ls.push_back(hs[kStLev + 2 * k]);
      le.push_back(hs[kStLev + 2 * k] + hs[kStLev + 2 * k + 1]);
    }
    l = hs[kStLevel];
    if (hs[kStStatus] == 1) {
      nlevels = l;
      done = true;
    } else if (hs[kStStatus] == 2) {
      bld.B.grow(2 * bld.B.cap + 4 * (size_t)kWgLevel, bld.nboxes);
    }
  };
  take_wg();
  while (!done && l < nlmax) {
    const int lo = ls[l], n = le[l] - ls[l];
    if (n <= kWgLevel && l + 1 <= pk[0]->d1 + pk[0]->d2) {
      hs[kStBoxes] = bld.nboxes;
      hs[kStLev + 2 * l] = lo;
      hs[kStLev + 2 * l + 1] = n;
      upload_bytes(state.p, hs.data(), sizeof(int) * kStWords, st);
      refine_wg(l);
      readback(hs.data(), state.p, sizeof(int) * kStWords, st);
      take_wg();
      continue;
    }
    // the batch: levels l .. l+K-1 refined, sizes bounded by ub[k]
    int K = std::min(kBatch, nlmax - l);
    if (pk[0]->d2 == 0 && l < d1) K = std::min(K, d1 - l);
    // as many levels as fit the capacity a batch may reserve
    const int64_t limit = std::max<int64_t>(kBatchBoxes, 2 * (int64_t)bld.nboxes);
    std::vector<int64_t> ub{n};
    int64_t reserve = 0;
    for (int k = 1; k <= K; ++k) {
      const int64_t u = std::min<int64_t>(4 * ub[k - 1], lev_cap);
      if (reserve + u > limit) {
        K = k - 1;
        break;
      }
      ub.push_back(u);
      reserve += u;
    }
    const bool batch = (pk[0]->d2 != 0 || l < d1) && K > 1;
    if (!batch) {
      // one level, exact (pts_tree2d.f:551-631 as written)
      bld.ensure_flag(n);
      launch1d(k_refine_flags, n, st, lo, bld.B.ses.p, bld.B.set.p, idivflag, ndiv, bld.flag.p);
      if (l + 1 > d1 && pk[0]->d2 == 0) {
        // a box at level d1 may need splitting: extend the paths (rare: only
        // for points closer than 2^-21 of the domain)
        if (bld.scan(n) > 0) {
          const int d2 = std::min(kD2Max, std::min(62, nlmax) - d1);
          pkx[0].build(src, ns, root[0], root[1], bsall[0], d1, d2, st);
          pkx[1].build(trg, nt, root[0], root[1], bsall[0], d1, d2, st);
          pk[0] = &pkx[0];
          pk[1] = &pkx[1];
          bld.ks = pk[0]->view();
          bld.kt = pk[1]->view();
        }
      }
      const int base = bld.nboxes;
      bs.push_back(bsall[l + 1]);
      const int nref = bld.refine(lo, n, bs[l + 1], l + 1, 0);
      if (nref == 0) {
        bs.pop_back();
        nlevels = l;
        break;
      }
      ls.push_back(base);
      le.push_back(bld.nboxes);
      ++l;
      continue;
    }
    bld.B.grow(bld.nboxes + (size_t)reserve, bld.nboxes);
    int64_t ubmax = 1;
    for (int k = 0; k < K; ++k) ubmax = std::max(ubmax, ub[k]);
    DBuf<int> part(ceil_div(ubmax, kRefTile), st);
    {
      const int h[2] = {lo, n};
      upload_bytes(dlev.p + 2 * l, h, sizeof(h), st);
      for (int k = 0; k < K; ++k) {
        const int L = l + k;
        const dim3 grid(ceil_div(ub[k], kRefTile));
        hipLaunchKernelGGL(k_lv_count, grid, dim3(kRefTile), 0, st, (const int*)dlev.p, L,
                           bld.B.ses.p, bld.B.set.p, idivflag, ndiv, part.p);
        hipLaunchKernelGGL(k_lv_children, grid, dim3(kRefTile), 0, st, dlev.p, L,
                           (const int*)part.p, idivflag, ndiv, 0.5 * bsall[L + 1],
                           bld.B.centers.p, bld.B.ilevel.p, bld.B.iparent.p, bld.B.nchild.p,
                           bld.B.ichild.p, bld.B.ses.p, bld.B.set.p, bld.B.iflag.p, bld.ks,
                           bld.kt);
        hip_throw(hipGetLastError(), "refine");
      }
      std::vector<int> hl(2 * (K + 1));
      readback(hl.data(), dlev.p + 2 * l, sizeof(int) * 2 * (K + 1), st);
      bld.nboxes = hl[2 * K] + hl[2 * K + 1];
      for (int k = 1; k <= K; ++k) {
        if (hl[2 * k + 1] == 0) {
          nlevels = l + k - 1;
          done = true;
          break;
        }
        bs.push_back(bsall[l + k]);
        ls.push_back(hl[2 * k]);
        le.push_back(hl[2 * k] + hl[2 * k + 1]);
      }
    }
    l += K;
  }
  ls.resize(nlevels + 1);
  le.resize(nlevels + 1);
  bs.resize(nlevels + 1);
  bld.computecoll(ls, le, bs, nlevels, state.p + kStBig);

  // ---- level restriction (pts_tree_fix_lr, pts_tree2d.f:758-1061); every
  // box's iflag is 0 here
  LevelTab T{};
  auto level_tab = [&]() {
    for (int k = 0; k <= nlevels; ++k) {
      T.ls[k] = ls[k];
      T.le[k] = le[k];
      T.bs[k] = bs[k];
    }
  };
  level_tab();
  std::vector<int> ts(nlevels + 2, 0), te(nlevels + 2, 0);
  int added = 0;
  DBuf<int> part;
  if (nlevels >= 2) {
    const int nb0 = bld.nboxes;
    {
      LevelReals dist{};
      for (int l = 2; l <= nlevels; ++l) dist.v[l] = 1.05 * (bs[l - 1] + bs[l - 2]) / 2.0;
      launch1d(k_flag1, le[nlevels] - ls[2], st, ls[2], dist, bld.B.ilevel.p, bld.B.iparent.p,
               bld.B.ncoll.p, bld.B.coll.p, bld.B.nchild.p, bld.B.centers.p, bld.B.iflag.p);
    }
    if (nb0 <= kWgBoxes) {
      for (;;) {
        hipLaunchKernelGGL(k_flags_wg, dim3(1), dim3(kWgThreads), 0, st, T, nlevels, nb0,
                           (int)std::min<size_t>(bld.B.cap, INT32_MAX), ptrs(bld.B), bld.ks,
                           bld.kt, state.p);
        hip_throw(hipGetLastError(), "level restriction");
        readback(hs.data(), state.p, sizeof(int) * kStWords, st);
        if (hs[kStStatus] == 0) break;
        bld.B.fit(5 * (size_t)nb0, nb0);
      }
      for (int l = 2; l <= nlevels - 1; ++l) {
        ts[l] = hs[kStLev + 2 * l];
        te[l] = hs[kStLev + 2 * l + 1];
      }
    } else {
      for (int k = 0; k < kStWords; ++k)
        if (k != kStBig) hs[k] = 0;
      upload_bytes(state.p, hs.data(), sizeof(int) * kStBig, st);
      upload_bytes(state.p + kStLev, hs.data() + kStLev, sizeof(int) * (kStWords - kStLev), st);
      for (int l = nlevels; l >= 1; --l) {
        const double distest = 1.05 * (bs[l] + bs[l - 1]) / 2.0;
        launch1d(k_flag2, le[l] - ls[l], st, ls[l], distest, bld.B.iparent.p, bld.B.ncoll.p,
                 bld.B.coll.p, bld.B.nchild.p, bld.B.centers.p, bld.B.iflag.p);
      }
      // the flags are fixed now: all levels refine together, with room for the
      // boxes that they make
      const int n = nlevels >= 3 ? le[nlevels - 2] - ls[1] : 0;
      part.alloc(ceil_div(std::max(n, 1), kLrTile), st);
      launch1d(k_flag_count, n, st, ls[1], (const int*)bld.B.iflag.p, (const int*)bld.B.ilevel.p,
               part.p, state.p);
      readback(hs.data(), state.p, sizeof(int) * kStWords, st);
      int64_t at = nb0;
      for (int l = 2; l <= nlevels - 1; ++l) {
        ts[l] = (int)at;
        at += 4 * (int64_t)hs[kStLev + 2 * l];
        if (at > INT32_MAX) throw HipError{hipErrorOutOfMemory, "tree boxes"};
        te[l] = (int)at;
      }
      if (at > nb0) {
        bld.B.fit((size_t)at, nb0);
        hipLaunchKernelGGL(k_flag_children<0>, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, ls[1],
                           0, nb0, (const int*)part.p, T,
                           (int)std::min<size_t>(bld.B.cap, INT32_MAX), ptrs(bld.B), bld.ks,
                           bld.kt, state.p);
        hip_throw(hipGetLastError(), "level restriction");
      }
    }
    for (int l = 2; l <= nlevels - 1; ++l) added += te[l] - ts[l];
    bld.nboxes += added;
  } else {
    readback(hs.data(), state.p, sizeof(int) * kStLev, st);
  }
  const bool big = hs[kStBig] != 0;
  // With no box added by the flagged refinement no box carries flag 3, the
  // updateflags sweep below refines nothing and both reorganisations are the
  // identity: the tree is already level-restricted.
  if (added > 0) {
    // the sweep over the levels, the new boxes' ranges kept on the device:
    // two launches a level and one round trip in all
    // (it adds 0.7 to 1.0 times what the flagged refinement added on curves and
    // clusters, 1.5 around isolated tight clusters, little where that added little)
    const int cap = (int)std::min<int64_t>(
        bld.nboxes + (int64_t)room * (13 * (int64_t)added / 8 + 64), INT32_MAX);
    bld.reorg(ls, le, ts, te, nlevels, (size_t)cap);
    bld.B.alloc_coll((size_t)cap);
    part.alloc((size_t)cap / kLrTile + 1, st);
    bld.computecoll(ls, le, bs, nlevels);
    level_tab();
    for (int k = 0; k < kStWords; ++k) hs[k] = 0;
    hs[kStLev + 2 * 2] = hs[kStLev + 2 * 2 + 1] = bld.nboxes;
    upload_bytes(state.p, hs.data(), sizeof(int) * kStWords, st);
    int64_t tail_ub = 0;
    for (int l = 2; l <= nlevels - 2; ++l) {
      const int n1 = le[l] - ls[l];
      const double distest = 1.05 * (bs[l] + bs[l + 1]) / 2.0;
      const unsigned n = (unsigned)(n1 + tail_ub);
      if (n > 0) {
        hipLaunchKernelGGL(k_sweep_flags, dim3(ceil_div(n, kLrTile)), dim3(256), 0, st, n1, ls[l],
                           l, (int)tail_ub, kColl * bs[l], distest, ptrs(bld.B), part.p, state.p);
        hipLaunchKernelGGL(k_flag_children<1>, dim3(ceil_div(n, 256)), dim3(256), 0, st, n1,
                           ls[l], l, 0, (const int*)part.p, T, cap, ptrs(bld.B), bld.ks, bld.kt,
                           state.p);
        hip_throw(hipGetLastError(), "level restriction");
      }
      tail_ub = std::min<int64_t>(
          std::min<int64_t>(4 * (int64_t)n, (int64_t)cap - bld.nboxes), (int64_t)262144 * room);
    }
    std::fill(ts.begin(), ts.end(), 0);
    std::fill(te.begin(), te.end(), 0);
    int added2 = 0;
    if (nlevels >= 4) {
      readback(hs.data(), state.p, sizeof(int) * kStWords, st);
      if (hs[kStStatus] != 0) return false;  // out of room
      for (int l = 3; l <= nlevels - 1; ++l) {
        ts[l] = hs[kStLev + 2 * l];
        te[l] = hs[kStLev + 2 * l + 1];
        added2 += te[l] - ts[l];
      }
      bld.nboxes += added2;
    }
    // the last level's tail has no colleagues yet; with nothing added the
    // second reorganisation is the identity and the colleagues are those
    // computed above
    if (added2 > 0) {
      bld.reorg(ls, le, ts, te, nlevels, (size_t)bld.nboxes);
      bld.computecoll(ls, le, bs, nlevels);
    }
  }

  // ---- final point order (pts_tree_sort, pts_tree2d.f:1222-1246)
  const int nb = bld.nboxes;
  t.nlevels = nlevels;
  t.nboxes = nb;
  t.lstart = ls;
  t.lend = le;
  t.boxsize = bs;
  t.isrc.alloc(std::max<int64_t>(ns, 1), st);
  t.itarg.alloc(std::max<int64_t>(nt, 1), st);
  t.leaf_s.alloc(std::max<int64_t>(ns, 1), st);
  t.leaf_t.alloc(std::max<int64_t>(nt, 1), st);
  DBuf<int>* perm[2] = {&t.isrc, &t.itarg};
  const int* se[2] = {bld.B.ses.p, bld.B.set.p};
  const int64_t npts[2] = {ns, nt};
  hipLaunchKernelGGL(k_leaf_of, dim3(ceil_div(nb, 256), nt > 0 ? 2 : 1), dim3(256), 0, st,
                     (int64_t)nb, bld.B.nchild.p, se[0], se[1], t.leaf_s.p, t.leaf_t.p);
  if (!big) {
    LeafOrder a;
    const int* leaf[2] = {t.leaf_s.p, t.leaf_t.p};
    for (int k = 0; k < 2; ++k) {
      a.n[k] = npts[k];
      a.leaf[k] = leaf[k];
      a.se[k] = se[k];
      a.perm[k] = pk[k]->perm.p;
      a.out[k] = perm[k]->p;
    }
    hipLaunchKernelGGL(k_leaf_rank, dim3(ceil_div(std::max(ns, nt), 256), nt > 0 ? 2 : 1),
                       dim3(256), 0, st, a);
  }
  hip_throw(hipGetLastError(), "point order");
  for (int k = 0; k < 2 && big; ++k) {
    if (npts[k] == 0) continue;
    // some leaf is too large to rank: stable sort of all points by leaf
    DBuf<unsigned long long> label(npts[k], st), lsorted(npts[k], st);
    launch1d(k_leaf_label, nb, st, bld.B.nchild.p, se[k], pk[k]->perm.p, label.p);
    int bits = 1;
    while ((int64_t(1) << bits) <= npts[k]) ++bits;
    // values: input indices 0..n-1 in input order
    radix_sort(label.p, lsorted.p, nullptr, perm[k]->p, npts[k], bits, st);
  }
  t.isrcse = std::move(bld.B.ses);
  t.itargse = std::move(bld.B.set);
  t.centers = std::move(bld.B.centers);
  t.ilevel = std::move(bld.B.ilevel);
  t.iparent = std::move(bld.B.iparent);
  t.nchild = std::move(bld.B.nchild);
  t.ichild = std::move(bld.B.ichild);
  t.ncoll = std::move(bld.B.ncoll);
  t.coll = std::move(bld.B.coll);
  return true;
}

void build_tree(const double* src, int64_t ns, const double* trg, int64_t nt, int ndiv,
                int idivflag, int nlmax, Tree& t, hipStream_t st, const TreePrep* prep) {
  if (nlmax > kMaxLevels) throw HipError{hipErrorInvalidValue, "nlmax beyond 51"};
  // bounding square, box sizes and sorted path keys: the caller's, or made here
  TreePrep own;
  const bool mine = !tree_prepare_matches(prep, src, ns, trg, nt, nlmax);
  if (mine) prepare_into(own, src, ns, trg, nt, nlmax, st);
  for (int room = 1;; room *= 4) {
    if (build_try(mine ? &own : prep, mine ? &own : nullptr, src, ns, trg, nt, ndiv, idivflag,
                  nlmax, t, st, room))
      return;
    if (room > 1 << 20) throw HipError{hipErrorOutOfMemory, "tree boxes"};
  }
}

// Points (sources + targets) held by the leaves of each level, levels beyond
// nbins - 1 counted in the last bin: per-block counts in LDS, then one global
// atomic per bin and block (integer counts, so the result does not depend on
// the order of the additions).
__global__ void k_leaf_hist(int64_t nb, const int* nchild, const int* ilevel, const int* ses,
                            const int* set, int nbins, unsigned long long* hist) {
  __shared__ unsigned long long h[kLeafHistMax];
  for (int k = threadIdx.x; k < nbins; k += blockDim.x) h[k] = 0;
  __syncthreads();
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b < nb && nchild[b] == 0) {
    const int n = (ses[2 * b + 1] - ses[2 * b]) + (set[2 * b + 1] - set[2 * b]);
    if (n > 0) atomicAdd(&h[min(ilevel[b], nbins - 1)], (unsigned long long)n);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < nbins; k += blockDim.x)
    if (h[k]) atomicAdd(&hist[k], h[k]);
}

// ---------------------------------------------------- key leaf histogram
// Leaf level of every point in the tree refined while a box holds more than
// ndiv sources (pts_tree_build's rule, common/pts_tree2d.f:551-631, without
// the level restriction of pts_tree_fix_lr), from the sorted source path
// keys alone: with w(j) = common levels of keys j and j + ndiv, the level-l box
// of a point holds more than ndiv sources iff some window j..j+ndiv of sorted
// sources lies in it -- for a source at sorted position i, iff w(j) >= l for a
// j in [i - ndiv, i]; for a target whose key sorts at position pos, iff
// min(w(j), common levels(key_j, target)) >= l for a j in [pos - ndiv - 1, pos].
// The leaf level is one more than the largest such l (0 if the root is a leaf).
__device__ __forceinline__ int key_common_levels(unsigned long long a, unsigned long long b,
                                                 int d1) {
  const unsigned long long x = a ^ b;
  if (x == 0) return d1;
  return (__clzll((long long)x) - (64 - 2 * d1)) >> 1;
}

__global__ void k_window_levels(int64_t m, int ndiv, int d1, const unsigned long long* keys,
                                unsigned char* w) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < m) w[j] = (unsigned char)key_common_levels(keys[j], keys[j + ndiv], d1);
}

// h[b] += the lanes of the wave that hold bin b (valid lanes only): one LDS
// add per distinct bin of the wave instead of one per lane
__device__ __forceinline__ void wave_bin_add(unsigned long long* h, bool valid, int b) {
  const int lane = threadIdx.x & 63;
  unsigned long long act = __ballot(valid);
  while (act) {  // uniform
    const int leader = __ffsll((long long)act) - 1;
    const int bl = __builtin_amdgcn_readlane(b, leader);
    const unsigned long long same = __ballot(valid && b == bl);
    if (lane == leader) atomicAdd(&h[bl], (unsigned long long)__popcll(same));
    act &= ~same;
  }
}

// Sources' leaf levels for ndiv <= kWinMax, kHistTile sorted keys per block of
// 256 threads.  Source i's leaf level is 1 + the largest w[j] =
// common levels(ks[j], ks[j + ndiv]) over the windows j in [i - ndiv, i]
// (0 outside [0, ns - ndiv - 1]): the maxima over ndiv + 1 consecutive w by
// doubling in LDS (after t passes m[x] = max w[x .. x + 2^t - 1]; the window
// is the union of two such ranges).
constexpr int kHistTile = 2048;
constexpr int kWinMax = 2048;
__global__ __launch_bounds__(256) void k_src_leaf_hist(int64_t ns, int ndiv, int d1,
                                                       const unsigned long long* __restrict__ ks,
                                                       int nbins, unsigned long long* hist) {
  __shared__ unsigned char m[kHistTile + kWinMax];
  __shared__ unsigned long long h[kLeafHistMax];
  for (int k = threadIdx.x; k < nbins; k += blockDim.x) h[k] = 0;
  const int64_t i0 = (int64_t)blockIdx.x * kHistTile;
  const int64_t last = ns - ndiv - 1;  // last window start
  const int len = kHistTile + ndiv;
  for (int x = threadIdx.x; x < len; x += 256) {
    const int64_t j = i0 - ndiv + x;
    m[x] = (j >= 0 && j <= last) ? (unsigned char)key_common_levels(ks[j], ks[j + ndiv], d1)
                                 : (unsigned char)0;
  }
  __syncthreads();
  constexpr int kPer = (kHistTile + kWinMax) / 256;
  int span = 1;
  while (2 * span <= ndiv + 1) {  // uniform
    unsigned char v[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int x = threadIdx.x + r * 256;
      v[r] = x < len ? m[x] : (unsigned char)0;
      if (x + span < len) v[r] = max(v[r], m[x + span]);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int x = threadIdx.x + r * 256;
      if (x < len) m[x] = v[r];
    }
    __syncthreads();
    span *= 2;
  }
  // span <= ndiv + 1 < 2 span: window [xi - ndiv, xi] = ranges from xi - ndiv and xi - span + 1
#pragma unroll
  for (int r = 0; r < kHistTile / 256; ++r) {
    const int64_t i = i0 + threadIdx.x + r * 256;
    const bool valid = i < ns;
    int b = 0;
    if (valid) {
      const int xi = (int)(i - i0) + ndiv;
      const int best = max((int)m[xi - ndiv], (int)m[xi - span + 1]);
      b = min(best + 1, nbins - 1);
    }
    wave_bin_add(h, valid, b);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < nbins; k += blockDim.x)
    if (h[k]) atomicAdd(&hist[k], h[k]);
}

// Leaf levels of the cnt points from i0 on (sources below ns, then targets) by
// direct window scans: the general path (targets; ndiv > kWinMax; ns <= ndiv).
__global__ void k_key_leaf_hist(int64_t cnt, int64_t i0, int64_t ns, int ndiv, int d1,
                                const unsigned long long* __restrict__ skeys,
                                const unsigned char* __restrict__ w,
                                const unsigned long long* __restrict__ tkeys, int nbins,
                                unsigned long long* hist) {
  __shared__ unsigned long long h[kLeafHistMax];
  for (int k = threadIdx.x; k < nbins; k += blockDim.x) h[k] = 0;
  __syncthreads();
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = i0 + g;
  int bin = 0;
  if (g < cnt) {
    int lev = 0;
    if (ns > ndiv) {
      const int64_t last = ns - ndiv - 1;  // last window start
      int best = 0;
      if (i < ns) {
        for (int64_t j = max((int64_t)0, i - ndiv); j <= min(i, last); ++j)
          best = max(best, (int)w[j]);
      } else {
        const unsigned long long t = tkeys[i - ns];
        int64_t lo = 0, hi = ns;  // pos = first sorted source key >= t
        while (lo < hi) {
          const int64_t mid = (lo + hi) >> 1;
          if (skeys[mid] < t) lo = mid + 1;
          else hi = mid;
        }
        for (int64_t j = max((int64_t)0, lo - ndiv - 1); j <= min(lo, last); ++j)
          best = max(best, min((int)w[j], key_common_levels(skeys[j], t, d1)));
      }
      lev = best + 1;
    }
    bin = min(lev, nbins - 1);
  }
  wave_bin_add(h, g < cnt, bin);
  __syncthreads();
  for (int k = threadIdx.x; k < nbins; k += blockDim.x)
    if (h[k]) atomicAdd(&hist[k], h[k]);
}

namespace {
// hist[l] from the sorted source keys ks and the target keys kt (any order),
// both of d1 levels
void hist_from_keys(const unsigned long long* ks, int64_t ns, const unsigned long long* kt,
                    int64_t nt, int d1, int ndiv, int nbins, double* hist, hipStream_t st) {
  DBuf<unsigned long long> d(nbins, st);
  d.zero();
  // sources by LDS window maxima when the window fits, the rest by scans
  const bool tiled = ns > ndiv && ndiv <= kWinMax;
  if (tiled)
    hipLaunchKernelGGL(k_src_leaf_hist, dim3((unsigned)ceil_div(ns, (int64_t)kHistTile)),
                       dim3(256), 0, st, ns, ndiv, d1, ks, nbins, d.p);
  const int64_t i0 = tiled ? ns : 0;
  if (ns + nt > i0) {
    const int64_t m = ns > ndiv ? ns - ndiv : 0;
    DBuf<unsigned char> w(std::max<int64_t>(m, 1), st);
    launch1d(k_window_levels, m, st, ndiv, d1, ks, w.p);
    launch1d(k_key_leaf_hist, ns + nt - i0, st, i0, ns, ndiv, d1, ks,
             (const unsigned char*)w.p, kt, nbins, d.p);
  }
  std::vector<unsigned long long> h(nbins);
  readback(h.data(), d.p, sizeof(unsigned long long) * nbins, st);
  for (int k = 0; k < nbins; ++k) hist[k] = (double)h[k];
}
}  // namespace

void key_leaf_histogram(const double* src, int64_t ns, const double* trg, int64_t nt, int ndiv,
                        int nbins, double* hist, double* boxsize0, hipStream_t st) {
  if (nbins < 1 || nbins > kLeafHistMax) throw HipError{hipErrorInvalidValue, "histogram bins"};
  // levels up to nbins - 1 tell every bin apart (the last bin takes the leaf
  // levels from nbins - 1 on): shorter keys, fewer sort passes
  const int d1 = std::max(1, std::min(kD1, nbins - 1));
  const int nb = (int)std::min<int64_t>(kRedBlocks, std::max<int64_t>(1, ceil_div(ns + nt, 256)));
  DBuf<double> part(4 * nb, st), bounds(4, st);
  DBuf<unsigned long long> k0(ns, st), ks(ns, st), kt(std::max<int64_t>(nt, 1), st);
  RsPlan rs;  // the targets' keys are used unsorted
  rs.init(ns, 0, 2 * d1, st);
  hipLaunchKernelGGL(k_bbox_partial, dim3(nb), dim3(256), 0, st, src, ns, trg, nt, part.p,
                     rs.words.p, (int64_t)rs.words.n);
  hipLaunchKernelGGL(k_keys_count,
                     dim3(rs_count_grid(std::max(ns, nt)), nt > 0 ? 2 : 1),
                     dim3(kRsCountThreads), 0, st, src, ns, trg, nt, (const double*)part.p, nb, d1, rs.npass,
                     k0.p, kt.p, rs.hist(0), bounds.p);
  hip_throw(hipGetLastError(), "path keys");
  const unsigned long long* ki[2] = {k0.p, nullptr};
  unsigned long long* ko[2] = {ks.p, nullptr};
  rs.sort(ki, ko, nullptr, nullptr, st);
  if (boxsize0) {
    double bb[4], cx, cy;
    readback(bb, bounds.p, sizeof(bb), st);
    root_square(bb, &cx, &cy, boxsize0);
  }
  hist_from_keys(ks.p, ns, kt.p, nt, d1, ndiv, nbins, hist, st);
}

void prepared_leaf_histogram(const TreePrep* P, int ndiv, int nbins, double* hist,
                             double* boxsize0, hipStream_t st) {
  if (nbins < 1 || nbins > kLeafHistMax) throw HipError{hipErrorInvalidValue, "histogram bins"};
  if (boxsize0) *boxsize0 = P->bsall[0];
  // the prepared keys hold min(kD1, nlmax) levels; every level from
  // nbins - 1 on falls in the last bin, so deeper keys give the same counts
  hist_from_keys(P->pk[0].k1.p, P->ns, P->pk[1].k1.p, P->nt, P->pk[0].d1, ndiv, nbins, hist, st);
}

void leaf_level_histogram(const Tree& t, int nbins, double* hist, hipStream_t st) {
  if (nbins < 1 || nbins > kLeafHistMax) throw HipError{hipErrorInvalidValue, "histogram bins"};
  DBuf<unsigned long long> d(nbins, st);
  d.zero();
  launch1d(k_leaf_hist, t.nboxes, st, t.nchild.p, t.ilevel.p, t.isrcse.p, t.itargse.p, nbins,
           d.p);
  std::vector<unsigned long long> h(nbins);
  readback(h.data(), d.p, sizeof(unsigned long long) * nbins, st);
  for (int k = 0; k < nbins; ++k) hist[k] = (double)h[k];
}

}  // namespace fmm2d
