// Helpers of wavefronts (64 lanes) and blocks: queue appends with one atomic per
// block, exchange through LDS within a wavefront, counter reductions and the
// claiming of work.
#ifndef MUONX_DEVICE_WAVE_H_
#define MUONX_DEVICE_WAVE_H_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "claim_plan.h"

namespace muonx {

// Appends a block's lanes with `want` to a queue: returns each such lane's index.
// NW wavefronts (blockDim.x = 64 * NW) reserve their entries with one atomic per
// block, in block order. Every thread of the block must call it (it synchronises
// the block); `sh` is NW + 1 words of shared memory.
template <int NW>
__device__ __forceinline__ uint32_t block_append(bool want, uint32_t *counter, uint32_t *sh) {
  const uint64_t m = __ballot(want);
  const int lane = int(__lane_id());
  const int w = int(threadIdx.x) >> 6;
  if (lane == 0) sh[w] = uint32_t(__popcll(m));
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) tot += sh[k];
    sh[NW] = tot ? atomicAdd(counter, tot) : 0u;
  }
  __syncthreads();
  uint32_t base = sh[NW];
  for (int k = 0; k < w; ++k) base += sh[k];
  __syncthreads();
  return base + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
}

// Orders a wavefront's LDS accesses before and after it, where its lanes
// exchange values through LDS words that no other wavefront touches.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Three appends of a block at once, one entry per lane for `want_a` and
// `want_b` and `cnt` for the third queue: three threads take the block's
// places together, so a block waits for one round of atomics instead of
// three. `sh` is used by this call only: callers in a loop alternate between
// two, so that the next call does not overwrite what a slower wavefront
// still reads (the call after it comes behind that wavefront's next barrier).
struct BlockAppend3 {
  static constexpr int kWaves = 8, kWords = 3 * (kWaves + 1);
  uint32_t a, b, c;
  __device__ __forceinline__ BlockAppend3(bool want_a, bool want_b, uint32_t cnt, uint32_t *ca, uint32_t *cb,
                                          uint32_t *cc, uint32_t *sh) {
    const int lane = int(__lane_id());
    const int w = int(threadIdx.x) >> 6;
    const uint64_t ma = __ballot(want_a), mb = __ballot(want_b), below = (1ull << lane) - 1ull;
    uint32_t incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t v = uint32_t(__shfl_up(int(incl), off));
      if (lane >= off) incl += v;
    }
    if (lane == 63) {
      sh[w] = uint32_t(__popcll(ma));
      sh[kWaves + w] = uint32_t(__popcll(mb));
      sh[2 * kWaves + w] = incl;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      uint32_t tot = 0;
#pragma unroll
      for (int k = 0; k < kWaves; ++k) tot += sh[threadIdx.x * kWaves + k];
      uint32_t *ctr = threadIdx.x == 0 ? ca : threadIdx.x == 1 ? cb : cc;
      sh[3 * kWaves + threadIdx.x] = tot ? atomicAdd(ctr, tot) : 0u;
    }
    __syncthreads();
    a = sh[3 * kWaves] + uint32_t(__popcll(ma & below));
    b = sh[3 * kWaves + 1] + uint32_t(__popcll(mb & below));
    c = sh[3 * kWaves + 2] + incl - cnt;
    for (int k = 0; k < w; ++k) {
      a += sh[k];
      b += sh[kWaves + k];
      c += sh[2 * kWaves + k];
    }
  }
};

__device__ __forceinline__ void wave_count(uint32_t n, unsigned long long *ctr) {
  unsigned long long a = n;
  for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off);
  if (__lane_id() == 0 && a) atomicAdd(ctr, a);
}

// Work claiming for kernels that give each lane a new item as soon as its
// current one is finished: the wavefront's ClaimPlan (claim_plan.h), the same
// in every lane.
struct WaveFetch {
  ClaimPlan p;
  __device__ __forceinline__ explicit WaveFetch(uint32_t items, uint32_t max_chunk = 256)
      : p(items, gridDim.x, gridDim.x * (blockDim.x >> 6),
          uint32_t(__builtin_amdgcn_readfirstlane(int(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)))),
          blockIdx.x, max_chunk) {}
  // Called by every lane of the wavefront with the ballot of `need`; returns
  // the index claimed for this lane (meaningful where `need` is set; an
  // index >= the item count means none is left).
  __device__ __forceinline__ uint32_t claim(uint64_t needm, uint32_t *counters) {
    const uint32_t lane = __lane_id();
    const uint32_t cnt = uint32_t(__popcll(needm));
    const uint32_t rank = uint32_t(__popcll(needm & ((1ull << lane) - 1ull)));
    const uint32_t rem = p.cend - p.cbase;
    uint32_t k;
    if (rem >= cnt) {
      k = p.cbase + rank;
      p.cbase += cnt;
    } else {
      uint32_t v = 0;
      if (p.counted()) {
        if (lane == 0) v = atomicAdd(counters + p.group * kClaimStride, 1u);
        v = uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
      }
      const uint32_t nb = p.next(v);
      k = rank < rem ? p.cbase + rank : nb + (rank - rem);
      p.cbase = nb + (cnt - rem);
      p.cend = nb + p.chunk;
    }
    return k;
  }
};

}  // namespace muonx

#endif
