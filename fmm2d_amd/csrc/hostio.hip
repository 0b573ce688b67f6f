// Small host <-> device transfers in stream order (devbuf.h: readback,
// upload_bytes).
//
// readback: a one-block kernel stores the words into pinned host memory and
// then, after a system-scope fence, a sequence number; the host polls for
// that number.  A copy into pageable memory followed by a stream
// synchronisation takes about 20 microseconds per round trip on MI355X, this
// about 6, and an FMM call makes dozens of such round trips (level counts,
// list sizes).  The pinned boxes are kept in a pool for the life of the
// process; one box serves one readback at a time.
//
// upload_bytes: the words travel in the arguments of a store kernel, which the
// runtime copies at launch, so no synchronisation keeps the host memory alive.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <vector>

#include "devbuf.h"
#include "stage_pool.h"

namespace fmm2d {

namespace {

constexpr int kBoxHead = 16;  // words before the data (the sequence number is word 0)

__global__ void k_readback(const unsigned* __restrict__ src, int nw,
                           const unsigned* __restrict__ src2, int nw2, unsigned* box,
                           unsigned seq) {
  for (int i = threadIdx.x; i < nw; i += blockDim.x) box[kBoxHead + i] = src[i];
  for (int i = threadIdx.x; i < nw2; i += blockDim.x) box[kBoxHead + nw + i] = src2[i];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(box, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int N> struct InlineWords {
  unsigned w[N];
};

template <int N>
__global__ void k_store_inline(unsigned* __restrict__ dst, int nw, InlineWords<N> a) {
  for (int i = threadIdx.x; i < nw; i += blockDim.x) dst[i] = a.w[i];
}

template <int N> void store_inline(void* dst, const void* src, size_t bytes, hipStream_t st) {
  InlineWords<N> a;
  std::memcpy(a.w, src, bytes);
  hipLaunchKernelGGL(k_store_inline<N>, dim3(1), dim3(256), 0, st, static_cast<unsigned*>(dst),
                     (int)(bytes / 4), a);
}

struct Box {
  unsigned* h = nullptr;  // pinned: [0] sequence number, [kBoxHead ..] data
  unsigned seq = 0;
};

std::mutex g_box_mu;
std::vector<Box*> g_boxes;  // free boxes (never returned to the runtime)

Box* box_acquire() {
  {
    std::lock_guard<std::mutex> g(g_box_mu);
    if (!g_boxes.empty()) {
      Box* b = g_boxes.back();
      g_boxes.pop_back();
      return b;
    }
  }
  void* p = nullptr;
  hip_throw(hipHostMalloc(&p, 4 * kBoxHead + kReadbackMax, hipHostMallocCoherent),
            "hipHostMalloc (readback box)");
  Box* b = new Box;
  b->h = static_cast<unsigned*>(p);
  __atomic_store_n(b->h, 0u, __ATOMIC_RELEASE);
  return b;
}

void box_release(Box* b) {
  std::lock_guard<std::mutex> g(g_box_mu);
  g_boxes.push_back(b);
}

}  // namespace

void readback(void* dst, const void* src, size_t bytes, hipStream_t st) {
  readback2(dst, src, bytes, nullptr, nullptr, 0, st);
}

void readback2(void* dst, const void* src, size_t bytes, void* dst2, const void* src2,
               size_t bytes2, hipStream_t st) {
  if (bytes + bytes2 == 0) return;
  if (bytes + bytes2 > kReadbackMax || bytes % 4 != 0 || bytes2 % 4 != 0) {
    if (bytes) hip_throw(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st), "copy");
    if (bytes2) hip_throw(hipMemcpyAsync(dst2, src2, bytes2, hipMemcpyDeviceToHost, st), "copy");
    hip_throw(hipStreamSynchronize(st), "sync");
    return;
  }
  AsyncRead r;
  r.begin(src, bytes, src2, bytes2, st);
  r.finish(dst, dst2);
}

AsyncRead::~AsyncRead() {
  // an unfinished read (an error in between): its kernel may still write the box
  if (!box) return;
  if (!done && hipStreamSynchronize(st) != hipSuccess) return;
  box_release(static_cast<Box*>(box));
}

void AsyncRead::begin(const void* src, size_t bytes, const void* src2, size_t bytes2,
                      hipStream_t s) {
  if (bytes + bytes2 > kReadbackMax || bytes % 4 != 0 || bytes2 % 4 != 0)
    throw HipError{hipErrorInvalidValue, "readback size"};
  Box* b = box_acquire();
  box = b;
  n1 = bytes;
  n2 = bytes2;
  st = s;
  if (++b->seq == 0) b->seq = 1;  // 0 is the initial word
  hipLaunchKernelGGL(k_readback, dim3(1), dim3(256), 0, st, static_cast<const unsigned*>(src),
                     (int)(bytes / 4), static_cast<const unsigned*>(src2), (int)(bytes2 / 4),
                     b->h, b->seq);
  hip_throw(hipGetLastError(), "readback launch");
}

bool AsyncRead::ready() const {
  const Box* b = static_cast<const Box*>(box);
  return __atomic_load_n(b->h, __ATOMIC_ACQUIRE) == b->seq;
}

void AsyncRead::finish(void* dst, void* dst2) {
  Box* b = static_cast<Box*>(box);
  // poll for up to 200 microseconds, then block on the stream (which also
  // reports a failure of the work queued before)
  const auto t0 = std::chrono::steady_clock::now();
  for (unsigned it = 1;; ++it) {
    if (__atomic_load_n(b->h, __ATOMIC_ACQUIRE) == b->seq) break;
    if ((it & 1023u) == 0 &&
        std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(200)) {
      hip_throw(hipStreamSynchronize(st), "sync");
      if (__atomic_load_n(b->h, __ATOMIC_ACQUIRE) != b->seq)
        throw HipError{hipErrorUnknown, "readback"};
      break;
    }
  }
  done = true;
  if (n1) std::memcpy(dst, b->h + kBoxHead, n1);
  if (n2) std::memcpy(dst2, b->h + kBoxHead + n1 / 4, n2);
}

namespace {

std::mutex g_stage_mu;
StagePool g_stage;

}  // namespace

void* Staging::get(size_t bytes, hipStream_t s) {
  st = s;
  {
    std::lock_guard<std::mutex> g(g_stage_mu);
    const StagePool::Buf b = g_stage.take(bytes);
    if (b.p) {
      p = b.p;
      cap = b.cap;
      return p;
    }
  }
  const size_t want = std::max(size_t(1) << 18, (bytes + (size_t(1) << 16)) >> 16 << 16);
  void* q = nullptr;
  hip_throw(hipHostMalloc(&q, want, hipHostMallocDefault), "hipHostMalloc (staging)");
  p = q;
  cap = want;
  return p;
}

Staging::~Staging() {
  if (!p) return;
  if (hipStreamSynchronize(st) != hipSuccess) return;  // a copy may still read it
  std::vector<StagePool::Buf> gone;
  bool kept = false;
  try {
    std::lock_guard<std::mutex> g(g_stage_mu);
    gone = g_stage.give(StagePool::Buf{p, cap});
    kept = true;
  } catch (...) {  // no memory for the pool's list
  }
  if (!kept) (void)hipHostFree(p);
  for (const StagePool::Buf& b : gone) (void)hipHostFree(b.p);
}

void staging_release() {
  std::vector<StagePool::Buf> all;
  {
    std::lock_guard<std::mutex> g(g_stage_mu);
    all.swap(g_stage.free);
  }
  for (const StagePool::Buf& b : all) (void)hipHostFree(b.p);
}

void upload_bytes(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return;
  if (bytes > kUploadInline || bytes % 4 != 0) {
    hip_throw(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st), "upload");
    hip_throw(hipStreamSynchronize(st), "sync");  // src may die after return
    return;
  }
  if (bytes <= 1024) store_inline<256>(dst, src, bytes, st);
  else store_inline<kUploadInline / 4>(dst, src, bytes, st);
  hip_throw(hipGetLastError(), "upload launch");
}

}  // namespace fmm2d
