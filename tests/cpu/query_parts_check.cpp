// Query launches (query_parts.h) on the CPU: the parts of a batch answer every
// ray once from its own coordinates, with indices of a launch held in a few bits
// as the kernels hold them in 32, and the part in use keeps 3 * ray + axis below
// 2^32 for any batch. Prints "ok".
#include <cstdio>
#include <vector>

#include "query_parts.h"

using namespace muonx;

// A kernel whose coordinate index wraps at 2^bits.
static bool Check(uint32_t n, uint32_t part, int bits, bool with_tmax, bool any) {
  std::vector<float> o(3 * size_t(n)), d(3 * size_t(n)), tmax(n), t(n, -1.0f);
  std::vector<int32_t> prim(n, -1);
  std::vector<uint8_t> occ(n, 0);
  for (size_t k = 0; k < o.size(); ++k) o[k] = float(k), d[k] = -float(k);
  for (uint32_t k = 0; k < n; ++k) tmax[k] = float(k) + 0.5f;
  const uint32_t mask = bits < 32 ? (1u << bits) - 1u : ~0u;
  bool ok = true;
  uint32_t seen = 0;
  const QueryArrays all{o.data(), d.data(), with_tmax ? tmax.data() : nullptr, any ? nullptr : prim.data(),
                        any ? nullptr : t.data(), any ? occ.data() : nullptr};
  const int rc = ForEachPart(all, n, part, [&](const QueryArrays &q, uint32_t m) {
    ok = ok && m > 0 && m <= part && (q.tmax != nullptr) == with_tmax && (q.occ != nullptr) == any;
    for (uint32_t i = 0; i < m; ++i, ++seen) {
      const float x = q.o[(3 * i) & mask], z = q.d[(3 * i + 2) & mask];
      ok = ok && x == float(3 * size_t(seen)) && z == -float(3 * size_t(seen) + 2);
      if (with_tmax) ok = ok && q.tmax[i] == float(seen) + 0.5f;
      if (any) ++q.occ[i];
      else ++q.prim[i], q.t[i] = x;
    }
    return 0;
  });
  ok = ok && rc == 0 && seen == n;
  for (uint32_t k = 0; k < n; ++k) ok = ok && (any ? occ[k] == 1 : prim[k] == 0 && t[k] == float(3 * size_t(k)));
  if (!ok) std::printf("n %u part %u\n", n, part);
  return ok;
}

int main() {
  bool ok = true;
  for (uint32_t part : {1u, 2u, 63u, 64u, 85u})  // 3 * 85 = 255 < 2^8
    for (uint32_t n : {0u, 1u, 2u, 62u, 63u, 64u, 65u, 84u, 85u, 86u, 170u, 171u, 1000u})
      for (int form = 0; form < 4; ++form) ok = Check(n, part, 8, form & 1, form & 2) && ok;
  // the part in use: indices and grid steps (at most 2^26 threads) in 32 bits, all rays of the largest batch
  ok = ok && 3ull * (kQueryPart - 1) + 2 < (1ull << 32) && uint64_t(kQueryPart) + (1ull << 26) < (1ull << 32);
  alignas(16) static float base[4];
  for (uint32_t n : {kQueryPart - 1, kQueryPart, kQueryPart + 1, 1431655766u, 1u << 31, ~0u}) {
    uint64_t sum = 0;
    uint32_t parts = 0;
    const QueryArrays q{base, base, nullptr, nullptr, nullptr, nullptr};
    ForEachPart(q, n, kQueryPart, [&](const QueryArrays &p, uint32_t m) {
      ok = ok && uintptr_t(p.o) - uintptr_t(base) == 12ull * sum && m <= kQueryPart;
      sum += m;
      return ++parts > 8 ? -1 : 0;
    });
    ok = ok && sum == n && parts == (uint64_t(n) + kQueryPart - 1) / kQueryPart;
  }
  // an error ends it
  uint32_t calls = 0;
  ok = ok && ForEachPart(QueryArrays{base, base, nullptr, nullptr, nullptr, nullptr}, 2, 1, [&](const QueryArrays &, uint32_t) {
    ++calls;
    return -3;
  }) == -3 && calls == 1;
  std::puts(ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
