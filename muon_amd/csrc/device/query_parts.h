// A query's arrays and their split into launches. Plain C++, so
// tests/cpu/query_parts_check.cpp runs it on the CPU.
#ifndef MUONX_DEVICE_QUERY_PARTS_H_
#define MUONX_DEVICE_QUERY_PARTS_H_

#include <cstddef>
#include <cstdint>

namespace muonx {

// The most rays of a launch: the kernels index the rays' coordinates (3 * ray + axis) and
// step over rays in 32 bits.
constexpr uint32_t kQueryPart = 1u << 30;

struct QueryArrays {
  const float *o, *d;   // 3 per ray
  const float *tmax;    // or null
  int32_t *prim;        // closest hit
  float *t;             // or null
  uint8_t *occ;         // any hit
  // The arrays from ray `k` on.
  QueryArrays from(uint32_t k) const {
    return QueryArrays{o + 3 * size_t(k),           d + 3 * size_t(k),     tmax ? tmax + k : nullptr,
                       prim ? prim + k : nullptr,   t ? t + k : nullptr,   occ ? occ + k : nullptr};
  }
};

// Calls launch(arrays, rays) for each part of at most `part` of the n rays, in
// order, until one returns an error.
template <class F>
int ForEachPart(const QueryArrays &a, uint32_t n, uint32_t part, F &&launch) {
  for (uint32_t at = 0; at < n;) {
    const uint32_t m = n - at < part ? n - at : part;
    const int rc = launch(a.from(at), m);
    if (rc != 0) return rc;
    at += m;
  }
  return 0;
}

}  // namespace muonx

#endif
