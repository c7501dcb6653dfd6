// ClaimPlan (claim_plan.h) on the CPU: wavefronts that ask for random numbers
// of items in a random order, as the kernels' lanes do, take every item
// exactly once, never touch a counter unless NeedsClaims says so, and stay
// below 2^32. Prints "ok".
#include <cstdio>
#include <random>
#include <vector>

#include "claim_plan.h"

using namespace muonx;

static std::mt19937_64 rng(5);

static bool Check(uint32_t items, uint32_t blocks, uint32_t wpb, uint32_t max_chunk) {
  const uint32_t waves = blocks * wpb;
  std::vector<ClaimPlan> plan;
  for (uint32_t w = 0; w < waves; ++w) plan.emplace_back(items, blocks, waves, w, w / wpb, max_chunk);
  std::vector<uint8_t> taken(items, 0);
  std::vector<uint32_t> counter(kClaimGroups, 0), open(waves, 64);  // lanes not told that none is left
  std::vector<uint32_t> alive(waves);
  for (uint32_t w = 0; w < waves; ++w) alive[w] = w;
  bool ok = true, counted = false;
  while (!alive.empty()) {
    const size_t at = rng() % alive.size();
    const uint32_t w = alive[at];
    ClaimPlan &p = plan[w];
    const uint32_t cnt = 1 + uint32_t(rng() % open[w]);
    // as WaveFetch::claim
    const uint32_t rem = p.cend - p.cbase;
    uint32_t first = p.cbase, nb = 0;
    if (rem >= cnt) {
      p.cbase += cnt;
    } else {
      uint32_t v = 0;
      if (p.counted()) {
        counted = true;
        v = counter[p.group]++;
      }
      nb = p.next(v);
      p.cbase = nb + (cnt - rem);
      p.cend = nb + p.chunk;
    }
    for (uint32_t r = 0; r < cnt; ++r) {
      const uint64_t k = rem >= cnt || r < rem ? uint64_t(first) + r : uint64_t(nb) + (r - rem);
      if (k >> 32) ok = false;
      if (k >= items) --open[w];
      else if (taken[size_t(k)]++) ok = false;
    }
    if (open[w] == 0) {
      alive[at] = alive.back();
      alive.pop_back();
    }
  }
  for (uint8_t t : taken) ok = ok && t == 1;
  if (counted && !NeedsClaims(items, waves)) ok = false;
  if (!ok) std::printf("items %u blocks %u waves/block %u max chunk %u\n", items, blocks, wpb, max_chunk);
  return ok;
}

int main() {
  bool ok = true;
  const uint32_t edge[] = {1, 2, 3, 63, 64, 65, 127, 128, 129, 2047, 2048, 2049, 4095, 4097, 8191, 131071, 131072, 131073};
  for (uint32_t n : edge)
    for (uint32_t blocks : {1u, 7u, 64u, 1024u}) ok = Check(n, blocks, 2, 64) && ok;
  for (uint32_t rounds = 1; rounds <= 6; ++rounds)  // around the change from static to claimed chunks
    for (int d = -1; d <= 1; ++d)
      for (uint32_t blocks : {8u, 129u}) ok = Check(uint32_t(int(rounds * blocks * 2 * kChunk) + d), blocks, 2, 256) && ok;
  for (int k = 0; k < 400; ++k)
    ok = Check(1 + uint32_t(rng() % 400000), 1 + uint32_t(rng() % 300), 1 + uint32_t(rng() % 4), (rng() & 1) ? 64 : 256) && ok;
  // the largest counts: no chunk starts past 2^32
  for (uint32_t waves : {2u, 8192u, 32768u}) {
    ClaimPlan p(1u << 31, waves / 2, waves, waves - 1, (waves - 1) / 2, 256);
    // a group's counter passes its last chunk by at most one per wavefront
    const uint64_t last = (uint64_t(1) << 31) / (uint64_t(p.groups) * p.chunk) + waves / p.groups;
    ok = ok && uint64_t(p.step) + (last * p.groups + p.groups) * p.chunk < (uint64_t(1) << 32);
  }
  std::puts(ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
