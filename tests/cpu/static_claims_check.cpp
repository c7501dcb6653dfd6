// ClaimPlan (claim_plan.h) of a launch without claim counters on the CPU: the
// wavefronts take every item exactly once and ask no counter, also where the
// same launch with counters would. Prints "ok".
#include <cstdio>
#include <vector>

#include "claim_plan.h"

using namespace muonx;

static bool Check(uint32_t items, uint32_t blocks, uint32_t wpb, uint32_t max_chunk) {
  const uint32_t waves = blocks * wpb;
  std::vector<uint8_t> taken(items, 0);
  bool ok = true;
  for (uint32_t w = 0; w < waves; ++w) {
    ClaimPlan p(items, blocks, waves, w, w / wpb, max_chunk, false);
    for (int rounds = 0;; ++rounds) {
      for (uint32_t k = p.cbase; k < p.cend && k < items; ++k) ok = ok && taken[k]++ == 0;
      if (p.counted() || rounds > 1000) return false;
      const uint32_t nb = p.next(0);
      if (nb >= items) break;
      p.cbase = nb;
      p.cend = nb + p.chunk;
    }
  }
  for (uint8_t t : taken) ok = ok && t == 1;
  return ok;
}

int main() {
  bool ok = true;
  for (uint32_t blocks : {1u, 7u, 8u, 129u, 3072u})
    for (uint32_t wpb : {1u, 2u})
      for (uint32_t chunk : {64u, 256u})
        for (uint32_t rounds : {1u, 3u, 4u, 5u, 9u})
          for (int d = -1; d <= 1; ++d) {
            const uint32_t n = uint32_t(int(rounds * blocks * wpb * kChunk) + d);
            if (n > 8000000u) continue;
            ok = Check(n, blocks, wpb, chunk) && ok;
          }
  for (uint32_t n : {1u, 2u, 63u, 65u}) ok = Check(n, 5, 2, 64) && ok;
  // the largest counts: the last wavefront's chunks stay below 2^32
  ClaimPlan p(1u << 31, 16384, 32768, 32767, 16383, 256, false);
  uint64_t at = p.cbase;
  while (!p.counted() && p.snext < p.send) {
    const uint32_t nb = p.next(0);
    ok = ok && nb > at;
    at = nb;
  }
  ok = ok && !p.counted() && at < (1ull << 31) && uint64_t(p.snext) < (1ull << 32);
  std::puts(ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
