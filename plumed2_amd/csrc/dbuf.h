// Device buffers that grow (host code only).
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <string>

#include "p2a_internal.h"

namespace p2a {

template <class T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  uint64_t gen = 0;  // allocations so far
  int reserve(size_t m) {
    if (m <= n && p) return P2A_OK;
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
    gen++;
    // 1/8 headroom: list sizes drift between rebuilds, and every regrowth
    // is a hipFree (which waits for the device) plus a hipMalloc
    size_t want = std::max<size_t>(m + m / 8, 1);
    if (hipMalloc((void**)&p, want * sizeof(T)) != hipSuccess) {
      p = nullptr;
      return fail(P2A_ERR_NOMEM, "hipMalloc of " + std::to_string(want * sizeof(T)) + " bytes failed");
    }
    n = want;
    return P2A_OK;
  }
  DBuf() = default;
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  ~DBuf() {
    if (p) (void)hipFree(p);
  }
};

// Something noted about what a buffer holds, which ends when the buffer is
// allocated again.  The address does not tell: the allocator may hand the freed
// one out again, over memory that holds anything past the old capacity.
struct Held {
  uint64_t gen = 0;
  template <class T>
  void note(const DBuf<T>& b) {
    gen = b.p ? b.gen : 0;
  }
  template <class T>
  bool of(const DBuf<T>& b) const {
    return gen != 0 && gen == b.gen;
  }
  void drop() { gen = 0; }
};

}  // namespace p2a
