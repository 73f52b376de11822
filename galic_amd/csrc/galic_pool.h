// galic_pool.h -- device memory of one call: many buffers carved from a few allocations.  Host
// code only; the allocator is a template argument (tests/test_device_pool.py runs it on the CPU).
#pragma once

#include <stddef.h>

#include <algorithm>
#include <vector>

namespace galic {

// A tree call has some thirty buffers, and an allocation and its release cost about 0.1 ms.  Each
// allocation holds what is asked for and room for the buffers that follow it: twice what the call
// has taken so far, 16 MiB at least, and at most kPoolExtra more than asked for (1e7 sources: 34.2
// ms a call with 1 GiB, 36.4 with 64 MiB).  Where memory is short the room is left out.  What was
// spare before then can still be what a later buffer lacks, so a call that did not fit is made
// again with `exact` set: every buffer an allocation of its own.
//
// Mem: Error get(void **, size_t), void put(void *), Error good(), bool is_short(Error) and
// forget(), which drops the runtime's record of the error just returned (it would otherwise be
// found by the next check of a kernel launch).
constexpr size_t kPoolExtra = (size_t)1 << 30;

template <class Mem>
struct DevPool {
  std::vector<void *> ptrs;
  char *at = nullptr;
  size_t left = 0, taken = 0;
  const bool exact;
  explicit DevPool(bool exact_ = false) : exact(exact_) {}
  DevPool(const DevPool &) = delete;
  DevPool &operator=(const DevPool &) = delete;
  template <typename T>
  typename Mem::Error alloc(T **p, size_t n) {
    const size_t bytes = (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255;
    if(bytes > left) {
      const size_t roomy = std::min(bytes + kPoolExtra, std::max<size_t>(2 * taken, (size_t)16 << 20));
      size_t want = exact ? bytes : std::max(bytes, roomy);
      void *q = nullptr;
      typename Mem::Error e = Mem::get(&q, want);
      if(e != Mem::good()) Mem::forget();
      if(Mem::is_short(e) && want > bytes) {
        e = Mem::get(&q, want = bytes);
        if(e != Mem::good()) Mem::forget();
      }
      if(e != Mem::good()) return e;
      ptrs.push_back(q);
      at = (char *)q;
      left = want;
      taken += want;
    }
    *p = (T *)at;
    at += bytes;
    left -= bytes;
    return Mem::good();
  }
  ~DevPool() {
    for(void *p : ptrs) Mem::put(p);
  }
};

// call(pool) with room to spare, and again with exact buffers where that was too much.
template <class Pool, class Call>
int with_pool(int short_status, Call call) {
  int rc;
  {
    Pool B;
    rc = call(B);
  }
  if(rc == short_status) {
    Pool B(true);
    rc = call(B);
  }
  return rc;
}

}  // namespace galic
