// Host copies between a caller's records and the pinned staging chunks of a
// handle (plain C++ with OpenMP, built with g++ and linked into librhllc_hip.so).
#pragma once

#include <cstddef>
#include <cstdint>

namespace rhllc_records {

// The 40-byte fields at offsets off_a and off_b (each skipped when < 0) of n
// records of `stride` bytes, to or from consecutive 40- or 80-byte entries.
void gather(const void *recs, int64_t stride, int64_t off_a, int64_t off_b, int64_t n, void *out);
void scatter(void *recs, int64_t stride, int64_t off_a, int64_t off_b, int64_t n, const void *in);

// memcpy over several threads.
void copy(void *dst, const void *src, size_t bytes);

// Fills an array on its first use.  alloc(&p), then fill(p); slot is set once
// both have returned 0, so a failure leaves it null for the next use to try
// again, with release(p) called if only fill failed.
template <typename T, typename Alloc, typename Fill, typename Release>
auto fill_once(T *&slot, Alloc alloc, Fill fill, Release release) -> decltype(alloc(&slot)) {
  if (slot) return decltype(alloc(&slot))(0);
  T *p = nullptr;
  auto e = alloc(&p);
  if (e != 0) return e;
  e = fill(p);
  if (e != 0) {
    release(p);
    return e;
  }
  slot = p;
  return e;
}

}  // namespace rhllc_records
