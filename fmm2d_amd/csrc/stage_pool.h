// A bounded pool of free buffers (hostio.hip: pinned staging memory), host code
// without HIP so that its rule can be tested by itself.
//
// take hands out the smallest buffer that fits.  give adds a buffer and returns
// those to be freed: the one given back longest ago goes first while there are
// more than kMost buffers or kBytes bytes.  The pool so holds what the latest
// calls used; one that kept the first buffers it was given, and turned later ones
// away, had every call with larger tables allocate and free pinned memory
// (which synchronises the device) for good after a batch of small calls.
#pragma once
#include <cstddef>
#include <vector>

namespace fmm2d {

struct StagePool {
  static constexpr size_t kMost = 16;                    // fmm2d_batch runs on up to 16 streams
  static constexpr size_t kBytes = size_t(64) << 20;
  struct Buf {
    void* p;
    size_t cap;
  };
  std::vector<Buf> free;  // in the order they were given back

  // A buffer of at least `bytes`, out of the pool; p null: none.
  Buf take(size_t bytes) {
    size_t best = free.size();
    for (size_t k = 0; k < free.size(); ++k)
      if (free[k].cap >= bytes && (best == free.size() || free[k].cap < free[best].cap)) best = k;
    if (best == free.size()) return Buf{nullptr, 0};
    const Buf b = free[best];
    free.erase(free.begin() + (std::ptrdiff_t)best);
    return b;
  }
  std::vector<Buf> give(Buf b) {
    std::vector<Buf> gone;
    gone.reserve(free.size() + 1);  // (an exception leaves the pool as it was)
    free.push_back(b);
    size_t sum = 0;
    for (const Buf& f : free) sum += f.cap;
    while (free.size() > kMost || sum > kBytes) {
      sum -= free.front().cap;
      gone.push_back(free.front());
      free.erase(free.begin());
    }
    return gone;
  }
};

}  // namespace fmm2d
