// parallel.h -- a static-partition parallel loop for the host-side table
// builders (site classification, reordering, neighbour checks).  Each worker
// takes one contiguous range, so per-range results can be combined in range
// order and the outcome does not depend on the thread count.
#pragma once

#include <algorithm>
#include <cstdint>
#include <memory>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

namespace hlb {

// Workers for n independent items: one for every `grain` items, up to 16.  A
// thread costs ~20 us to start, the items of a default grain ~500 us to do.
constexpr int64_t kGrain = 16384;
inline int host_workers(int64_t n, int64_t grain = kGrain) {
  const int64_t hc = std::max(1u, std::thread::hardware_concurrency());
  return (int)std::max<int64_t>(1, std::min<int64_t>({16, hc, n / grain}));
}

// Calls body(w, lo, hi) for worker w over [lo, hi), the w-th of nw
// contiguous ranges of [0, n); returns nw.
template <typename F>
int parallel_ranges(int64_t n, F&& body, int64_t grain = kGrain) {
  const int nw = host_workers(n, grain);
  if (nw == 1) {
    body(0, int64_t(0), n);
    return 1;
  }
  std::vector<std::thread> pool;
  pool.reserve((size_t)nw);
  for (int w = 1; w < nw; ++w) {
    try {
      pool.emplace_back([&, w] { body(w, n * w / nw, n * (w + 1) / nw); });
    } catch (const std::system_error&) {
      body(w, n * w / nw, n * (w + 1) / nw);  // no thread to be had: here, then
    }
  }
  body(0, int64_t(0), n / nw);
  for (auto& t : pool) t.join();
  return nw;
}

// Vector elements left uninitialised by resize, for arrays that a parallel
// loop fills: the filling threads touch the pages first.
template <typename T>
struct RawAllocator : std::allocator<T> {
  template <typename U>
  struct rebind {
    using other = RawAllocator<U>;
  };
  template <typename U>
  void construct(U* p) noexcept {
    ::new ((void*)p) U;
  }
  template <typename U, typename... Args>
  void construct(U* p, Args&&... args) {
    ::new ((void*)p) U(std::forward<Args>(args)...);
  }
};
template <typename T>
using RawVector = std::vector<T, RawAllocator<T>>;

}  // namespace hlb
