// Engine capacities (engine_plan.h) on the CPU: at every capacity that
// EngineCapacityOk admits, the position of each queued path differs from
// kPathEnds and leaves the flags alone, and the last shadow slot fits its 32-bit
// index. Prints "ok".
#include <cstdio>
#include <initializer_list>

#include "engine_plan.h"

using namespace muonx;

int main() {
  bool ok = (kPathNextMask & (kPathHasMis | kPathHasShadow)) == 0;
  const uint64_t edge = 1ull << 30;
  for (uint64_t cap : {uint64_t(1), uint64_t(1024), edge / 4, edge / 2, edge - 2, edge - 1, edge, edge + 1, 2 * edge})
    for (uint64_t kmax : {1u, 2u, 3u, 4u, 130u}) {
      const bool admitted = EngineCapacityOk(cap, kmax);
      const bool fits = cap - 1 < kPathEnds && ((cap - 1) & ~uint64_t(kPathNextMask)) == 0 && cap * kmax <= (1ull << 31);
      if (admitted != fits) {
        std::printf("capacity %llu x %llu: %s\n", (unsigned long long)cap, (unsigned long long)kmax, admitted ? "admitted" : "refused");
        ok = false;
      }
      if (admitted) ok = ok && uint64_t(ShadowSlot(uint32_t(kmax) - 1, uint32_t(cap), uint32_t(cap) - 1)) == cap * kmax - 1;
    }
  ok = ok && EngineCapacityOk(edge - 1, 2) && !EngineCapacityOk(edge, 1);
  std::puts(ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
