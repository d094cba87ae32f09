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

}  // namespace rhllc_records
