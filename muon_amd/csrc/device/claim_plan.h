// Which items each wavefront of a work-claiming kernel takes (wave.h): plain
// index arithmetic, no HIP types, so tests/cpu/claim_plan_check.cpp runs it on
// the CPU.
#ifndef MUONX_DEVICE_CLAIM_PLAN_H_
#define MUONX_DEVICE_CLAIM_PLAN_H_

#include <cstddef>
#include <cstdint>

namespace muonx {

// Work claiming for kernels that give each lane a new item as soon as its
// current one is finished. Items are handed to wavefronts in chunks of 64 or
// more consecutive indices; wavefront w starts with chunk w, and then
//  * up to kStaticRounds chunks per wavefront: takes every waves-th chunk, with
//    no counter (NeedsClaims tells the host, which then need not clear one);
//  * beyond: claims chunks (then of up to max_chunk items, about four per
//    wavefront) from one of up to kClaimGroups counters, each handing out
//    every 16th chunk. Groups are made of eight consecutive blocks,
//    one on each XCD, so that a slower XCD takes fewer chunks of every group.
// A captured launch, whose replays no clear or order between streams would
// cover, stays within UnclaimedItems.
// Atomics on one address take 11.3 ns each here however few wavefronts are
// left (1.8 ns spread over 8 addresses, 0.24 over 64), so one counter bounds
// a launch by its chunks: 3,000,017 any-hit rays on 10,000 spheres take 677 us
// with one counter and 393 us with 16 (8 or 32: 402 / 397), 10^6 closest hits
// on the Cornell box 224 us with one and 76 us static, 2^24 on the level-7
// icosphere 2.59 and 2.54 ms (all static 3.03 ms: XCDs differ).
//
// Fewer items than lanes are spread over two wavefronts per SIMD of the whole
// card's 256 CUs (on fewer CUs over all of the grid's wavefronts) before a
// wavefront gets all of its lanes an item: a wavefront takes as long as the
// longest of its lanes at every step, and idle SIMDs cost nothing. 10,000
// exact closest hits on the level-5 icosphere take 95 us against 128 us with
// 64 rays to each wavefront, 1000 on the Cornell box 18 against 34 us; at
// least 2, 4, 8 or 16 rays each: 95 / 94 / 102 / 113 and 18 / 21 / 27 / 34 us;
// 1024, 2048, 4096 or 6144 wavefronts: within 1 % but for 200,000 any-hit
// rays, which 6144 make 16 % slower.
constexpr uint32_t kChunk = 64, kStaticRounds = 4, kClaimGroups = 16;
constexpr uint32_t kClaimStride = 64;  // counters on 256-byte lines of their own
constexpr size_t kClaimBytes = size_t(kClaimGroups) * kClaimStride * sizeof(uint32_t);
constexpr uint32_t kSpreadWaves = 2048, kSpreadMin = 2;

// The most items that `waves` wavefronts take without a counter.
constexpr uint64_t UnclaimedItems(uint32_t waves) { return uint64_t(waves) * kChunk * kStaticRounds; }
constexpr bool NeedsClaims(uint32_t items, uint32_t waves) { return items > UnclaimedItems(waves); }
// Items in a wavefront's first chunk.
constexpr uint32_t FirstChunk(uint32_t items, uint32_t waves) {
  const uint32_t each = items / (waves < kSpreadWaves ? waves : kSpreadWaves) + 1u;
  return each >= kChunk ? kChunk : (each < kSpreadMin ? kSpreadMin : each);
}

// Blocks of `wpb` wavefronts for a grid of at most `max_blocks`: as many as hold
// a wavefront with a first chunk.
constexpr uint32_t ClaimBlocks(uint64_t items, uint32_t max_blocks, uint32_t wpb) {
  const uint64_t waves =
      items / FirstChunk(items < 0xffffffffull ? uint32_t(items) : 0xffffffffu, max_blocks * wpb) + 1;
  const uint64_t blocks = (waves + wpb - 1) / wpb;
  return blocks < max_blocks ? uint32_t(blocks) : max_blocks;
}

// One wavefront's share: the chunk in hand and where the next one comes from.
// Item counts up to 2^31, at most 2^20 wavefronts.
struct ClaimPlan {
  static constexpr uint32_t kNone = 0x80000000u;  // past every item
  uint32_t cbase, cend;        // what is left of the chunk in hand
  uint32_t snext, send, step;  // static chunks: the next one's start, their end, their distance
  uint32_t group, groups;      // claimed chunks: the counter and their number, 0 for none,
  uint32_t chunk;              // the items of each
  constexpr ClaimPlan(uint32_t items, uint32_t blocks, uint32_t waves, uint32_t wave, uint32_t block,
                      uint32_t max_chunk)
      : cbase(0), cend(0), snext(0), send(0), step(0), group(0), groups(0), chunk(kChunk) {
    if (NeedsClaims(items, waves)) {
      groups = (blocks + 7u) / 8u < kClaimGroups ? (blocks + 7u) / 8u : kClaimGroups;  // none without blocks
      group = (block >> 3) % groups;
      const uint32_t c = (items / (4u * waves)) & ~63u;
      chunk = c < max_chunk ? c : max_chunk;
      cbase = wave * chunk;
      cend = cbase + chunk;
      step = waves * chunk;
      snext = send = step;
    } else {
      const uint32_t first = FirstChunk(items, waves);
      cbase = wave * first;
      cend = cbase + first;
      step = waves * kChunk;
      snext = first < kChunk ? items : cbase + step;  // one chunk each when spread
      send = items;
    }
  }
  // Whether the next chunk is the counter's to give.
  constexpr bool counted() const { return snext >= send && groups != 0u; }
  // Start of the next chunk; `v` is what the group's counter held (counted()).
  constexpr uint32_t next(uint32_t v) {
    if (counted()) return step + (v * groups + group) * chunk;
    if (snext >= send) return kNone;
    const uint32_t nb = snext;
    snext += step;
    return nb;
  }
};

}  // namespace muonx

#endif
