// Batched closest-hit / any-hit queries over device-resident rays
// (muonx_intersect_closest / muonx_intersect_any).
#include "exact_trace.h"
#include "query.h"
#include "query_parts.h"
#include "runtime.h"
#include "trace.h"
#include "traverse_launch.h"
#include "wave.h"

#include <mutex>
#include <string>

namespace muonx {

constexpr uint32_t kWavesPerBlock = kQueryBlock / 64;
template <int KIND, bool WW, int WIDTH, bool ANY, bool COUNT>
__global__ void __launch_bounds__(kQueryBlock) k_query(DevSceneView s, StackArgs sa, const float *__restrict__ ro,
                                                       const float *__restrict__ rd, const float *__restrict__ tmax,
                                                       uint32_t n, int32_t *__restrict__ prim_out,
                                                       float *__restrict__ t_out, uint8_t *__restrict__ occ_out,
                                                       unsigned long long *__restrict__ counters) {
  __shared__ uint2 lds[StackOf<KIND>::kLds * kQueryBlock];
  uint2 old[StackOf<KIND>::kPrivate];
  TraceCounters cnt{0, 0};
  for (uint32_t i = blockIdx.x * kQueryBlock + threadIdx.x; i < n; i += gridDim.x * kQueryBlock) {
    const V3 o{ro[3 * i], ro[3 * i + 1], ro[3 * i + 2]};
    const V3 d{rd[3 * i], rd[3 * i + 1], rd[3 * i + 2]};
    float best = tmax ? tmax[i] : __builtin_inff();
    const TraceRay r = make_ray(o, d);
    auto st = make_stack<KIND>(lds, kQueryBlock, sa, old);
    const int32_t p = trace_fast<WIDTH, ANY, COUNT, WW>(s, r, best, st, cnt);
    if (ANY) {
      occ_out[i] = p >= 0 ? 1 : 0;
    } else {
      prim_out[i] = p >= 0 ? s.prim_id[p] : -1;
      if (t_out) t_out[i] = p >= 0 ? best : 0.0f;
    }
  }
  if (COUNT) {
    // wave-level reduction, one atomic per wave
    unsigned long long a = cnt.nodes, b = cnt.prims;
    for (int off = 32; off > 0; off >>= 1) {
      a += __shfl_down(a, off);
      b += __shfl_down(b, off);
    }
    if ((threadIdx.x & 63) == 0) {
      atomicAdd(&counters[0], a);
      atomicAdd(&counters[1], b);
    }
  }
}

// Fast mode with per-lane ray fetch: a lane whose ray is finished takes the
// next unclaimed ray once at least `fetch_min` lanes of its wavefront are
// idle, so long rays no longer hold idle lanes (claims: WaveFetch).
template <int KIND, int WIDTH, bool ANY, bool COUNT>
__global__ void __launch_bounds__(kQueryBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
    k_query_dyn(DevSceneView s, StackArgs sa, const float *__restrict__ ro, const float *__restrict__ rd,
                const float *__restrict__ tmax, uint32_t n, int32_t *__restrict__ prim_out, float *__restrict__ t_out,
                uint8_t *__restrict__ occ_out, unsigned long long *__restrict__ counters, uint32_t *next,
                int fetch_min) {
  __shared__ uint2 lds[StackOf<KIND>::kLds * kQueryBlock];
  uint2 old[StackOf<KIND>::kPrivate];
  TraceCounters cnt{0, 0};
  auto st = make_stack<KIND>(lds, kQueryBlock, sa, old);
  LaneTrace<WIDTH, ANY, COUNT> lt;
  uint32_t idx = 0;
  WaveFetch wf(n, kChunk);
  bool walking = false, have = false, drained = false;
  while (true) {
    const uint64_t needm = __builtin_amdgcn_ballot_w64(!have && !drained);
    if (needm) {
      const uint32_t k = wf.claim(needm, next);
      if (!have && !drained) {
        if (k < n) {
          idx = k;
          const V3 o{ro[3 * k], ro[3 * k + 1], ro[3 * k + 2]};
          const V3 d{rd[3 * k], rd[3 * k + 1], rd[3 * k + 2]};
          lt.start(make_ray(o, d), tmax ? tmax[k] : __builtin_inff(), st);
          walking = have = true;
        } else {
          drained = true;
        }
      }
    }
    if (__builtin_amdgcn_ballot_w64(have) == 0) break;
    run_walks(s, lt, walking, st, cnt, __builtin_amdgcn_ballot_w64(drained) ? 65 : fetch_min);
    if (have && !walking) {
      have = false;
      if (ANY) {
        occ_out[idx] = lt.hit >= 0 ? 1 : 0;
      } else {
        prim_out[idx] = lt.hit >= 0 ? s.prim_id[lt.hit] : -1;
        if (t_out) t_out[idx] = lt.hit >= 0 ? lt.best : 0.0f;
      }
    }
  }
  if (COUNT) {
    wave_count(cnt.nodes, &counters[0]);
    wave_count(cnt.prims, &counters[1]);
  }
}

// Exact mode: the walks of a wavefront's lanes, each lane taking the next
// unclaimed ray once kExactRefill of them are idle. Bound by instruction
// issue (lanes 27-31 % used, 200 wavefront instructions per ray). Against one
// ray per lane and grid step, a node or a leaf step per iteration and the
// whole stack in LDS (three wavefronts per SIMD, now seven): 300,007
// incoherent rays on the level-6 icosphere 361 -> 259 us, 10^6 on 10,000
// spheres 1154 -> 391 us together with the reciprocal quotients. Refilling
// at 16, 32 or 48 idle lanes measured the same.
// Without PRIVATE the whole stack is in LDS (three wavefronts per SIMD at most):
// for calls that may not take private memory from the runtime.
constexpr int kExactRefill = 32;
template <int CAP, bool PRIVATE>
struct ExactStack {
  using T = PrivateStack<CAP>;
  static constexpr int kLds = kPrivateRing, kOld = T::kOld;
  static __device__ __forceinline__ T make(uint2 *lds, uint2 *old) { return T(lds + threadIdx.x, kQueryBlock, old); }
};
template <int CAP>
struct ExactStack<CAP, false> {
  using T = LdsStack<CAP>;
  static constexpr int kLds = CAP, kOld = 1;
  static __device__ __forceinline__ T make(uint2 *lds, uint2 *) { return T(lds + threadIdx.x, kQueryBlock); }
};
template <int CAP, bool PRIVATE, bool ANY, bool COUNT>
__global__ void __launch_bounds__(kQueryBlock)
    k_query_exact(DevSceneView s, const float *__restrict__ ro, const float *__restrict__ rd,
                  const float *__restrict__ tmax, uint32_t n, int32_t *__restrict__ prim_out,
                  float *__restrict__ t_out, uint8_t *__restrict__ occ_out, unsigned long long *__restrict__ counters,
                  uint32_t *next) {
  using Stack = ExactStack<CAP, PRIVATE>;
  __shared__ uint2 lds[Stack::kLds * kQueryBlock];
  uint2 old[Stack::kOld];
  auto st = Stack::make(lds, old);
  ExactWalk<COUNT, ANY ? kWalkAny : kWalkClosest> w;
  TraceCounters cnt;
  WaveFetch wf(n, kChunk);
  uint32_t idx = 0;
  bool walking = false, have = false, drained = false;
  while (true) {
    const uint64_t needm = __builtin_amdgcn_ballot_w64(!have && !drained);
    if (needm) {
      const uint32_t k = wf.claim(needm, next);
      if (!have && !drained) {
        if (k < n) {
          idx = k;
          have = true;
          const V3 o{ro[3 * k], ro[3 * k + 1], ro[3 * k + 2]};
          const V3 d{rd[3 * k], rd[3 * k + 1], rd[3 * k + 2]};
          walking = w.start(s, make_ray(o, d), tmax ? tmax[k] : __builtin_inff(), ANY, st, cnt);
        } else {
          drained = true;
        }
      }
    }
    if (__builtin_amdgcn_ballot_w64(have) == 0) break;
    run_walks(s, w, walking, st, cnt, __builtin_amdgcn_ballot_w64(drained) ? 65 : kExactRefill);
    if (have && !walking) {
      have = false;
      if (ANY) {
        occ_out[idx] = w.hit >= 0 ? 1 : 0;
      } else {
        prim_out[idx] = w.hit >= 0 ? s.prim_id[w.hit] : -1;
        if (t_out) t_out[idx] = w.hit >= 0 ? w.best : 0.0f;
      }
    }
  }
  if (COUNT) {
    wave_count(cnt.nodes, &counters[0]);
    wave_count(cnt.prims, &counters[1]);
  }
}

namespace {
template <bool ANY, bool COUNT>
struct QueryDynLaunch {
  const TraverseCfg &cfg;
  const DevSceneView &s;
  const QueryArrays &q;
  uint32_t n;
  unsigned long long *counters;
  uint32_t *next;
  int fetch_min;
  hipStream_t stream;
  template <int KIND, bool WW, int WIDTH>
  void run() const {
    const StackArgs sa{cfg.spill, cfg.gcap};
    hipLaunchKernelGGL((k_query_dyn<KIND, WIDTH, ANY, COUNT>), dim3(cfg.grid), dim3(kQueryBlock), 0, stream, s, sa,
                       q.o, q.d, q.tmax, n, q.prim, q.t, q.occ, counters, next, fetch_min);
  }
};

template <bool ANY, bool COUNT>
struct QueryLaunch {
  const TraverseCfg &cfg;
  const DevSceneView &s;
  const QueryArrays &q;
  uint32_t n;
  unsigned long long *counters;
  hipStream_t stream;
  template <int KIND, bool WW, int WIDTH>
  void run() const {
    const StackArgs sa{cfg.spill, cfg.gcap};
    hipLaunchKernelGGL((k_query<KIND, WW, WIDTH, ANY, COUNT>), dim3(cfg.grid), dim3(kQueryBlock), 0, stream,
                       s, sa, q.o, q.d, q.tmax, n, q.prim, q.t, q.occ, counters);
  }
};
}  // namespace

// Static scratch of muonx_intersect_noalloc: the claim counters of the
// per-lane fetch kernels (the first kClaimBytes) and the traversal stacks'
// spill region (the rest). Every GPU holds its own copy until the process
// ends; its device address is looked up once per device by
// InitStaticScratch (with the device current), never used by name on the
// host.
constexpr size_t kStaticScratchBytes = size_t(32) << 20;
constexpr size_t kStaticScratchHead = kClaimBytes;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxScratchDevices] = {};

void *StaticScratch(int device) {
  if (device < 0 || device >= kMaxScratchDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

__global__ void k_clear_claims(uint32_t *p) { p[threadIdx.x * kClaimStride] = 0u; }
}  // namespace

int InitStaticScratch(int device) {
  if (device < 0 || device >= kMaxScratchDevices) {
    SetError("static scratch: device index " + std::to_string(device) + " above the table of " +
             std::to_string(kMaxScratchDevices));
    return MUONX_ERR_INVALID;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return MUONX_OK;
  void *p = nullptr;
  MX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = p;
  return MUONX_OK;
}

// The claim counters of the per-lane fetch kernels, cleared on `stream`: in
// the static scratch with `noalloc` (by a kernel rather than a memset node),
// else in the context, ordered after its previous user like the spill region.
static int ClearClaims(muonx_ctx *ctx, hipStream_t stream, bool noalloc, void *scratch_base, uint32_t **next) {
  if (noalloc) {
    *next = static_cast<uint32_t *>(scratch_base);
    hipLaunchKernelGGL(k_clear_claims, dim3(1), dim3(kClaimGroups), 0, stream, *next);
    return MUONX_OK;
  }
  MX_HIP(ctx->fetch_ctr.Reserve(kClaimBytes));
  if (!ctx->spill_done) MX_HIP(hipEventCreateWithFlags(&ctx->spill_done, hipEventDisableTiming));
  MX_HIP(hipStreamWaitEvent(stream, ctx->spill_done, 0));
  MX_HIP(hipMemsetAsync(ctx->fetch_ctr.ptr, 0, kClaimBytes, stream));
  *next = ctx->fetch_ctr.as<uint32_t>();
  return MUONX_OK;
}

// Calls launch(arrays, rays, counters) for n rays on `waves` wavefronts, with
// cleared claim counters (else null) where they need them; `counted` says whether
// the context's were used. Under capture the rays go out in parts that need none:
// on replays after the first a recorded memset has left the counters as they
// were, and no replay waits for the context's other calls.
template <class F>
static int LaunchClaiming(muonx_ctx *ctx, const QueryArrays &q, uint32_t n, uint32_t waves, hipStream_t stream,
                          bool noalloc, void *scratch_base, bool *counted, F &&launch) {
  *counted = false;
  uint32_t *next = nullptr;
  if (NeedsClaims(n, waves)) {
    bool capturing = false;
    int rc = noalloc ? MUONX_OK : IsCapturing(stream, &capturing);
    if (rc != MUONX_OK) return rc;
    if (capturing)
      return ForEachPart(q, n, uint32_t(UnclaimedItems(waves)), [&](const QueryArrays &part, uint32_t m) {
        launch(part, m, next);
        return MUONX_OK;
      });
    if ((rc = ClearClaims(ctx, stream, noalloc, scratch_base, &next)) != MUONX_OK) return rc;
    *counted = !noalloc;
  }
  launch(q, n, next);
  return MUONX_OK;
}

// Exact mode: stacks in LDS and private memory (`noalloc`: in LDS alone), so the
// claim counters are the only scratch, and a batch without claims needs none.
// 6, 8, 12 or 16 blocks per CU: 308 / 301 / 260 / 260 us for 300,007 rays on the
// level-6 icosphere; with whole stacks in LDS, as many as its LDS holds.
constexpr int kExactBlocksPerCu = 12;
constexpr int kLdsBytes = 160 << 10;  // of a CU
static int LaunchExactQuery(muonx_ctx *ctx, const DevSceneView &s, bool any, const QueryArrays &q, uint32_t n,
                            unsigned long long *counters, hipStream_t stream, bool noalloc, void *scratch_base) {
  if (s.bvh_depth > 96) {
    SetError("BVH depth " + std::to_string(s.bvh_depth) + " exceeds the exact-mode traversal stack (96)");
    return MUONX_ERR_CAPACITY;
  }
  const int cap = s.bvh_depth <= 24 ? 24 : s.bvh_depth <= 48 ? 48 : 96;
  const int per_cu = noalloc ? std::min(kExactBlocksPerCu, kLdsBytes / (cap * kQueryBlock * int(sizeof(uint2))))
                             : kExactBlocksPerCu;
  const uint32_t cus = uint32_t(ctx->num_cus > 0 ? ctx->num_cus : 256);
  const uint32_t grid = ClaimBlocks(n, cus * uint32_t(per_cu), kWavesPerBlock);
  const auto launch = [&](const QueryArrays &q, uint32_t m, uint32_t *next) {
#define MX_QX(CAP, P, A, C) \
  hipLaunchKernelGGL((k_query_exact<CAP, P, A, C>), dim3(grid), dim3(kQueryBlock), 0, stream, s, q.o, q.d, q.tmax, m, \
                     q.prim, q.t, q.occ, counters, next)
#define MX_QXP(CAP, A, C) \
  if (noalloc) MX_QX(CAP, false, A, C); \
  else MX_QX(CAP, true, A, C)
#define MX_QXC(A, C) \
  if (cap == 24) { MX_QXP(24, A, C); } \
  else if (cap == 48) { MX_QXP(48, A, C); } \
  else { MX_QXP(96, A, C); }
    if (any) {
      MX_QXC(true, false);
    } else if (counters) {
      MX_QXC(false, true);
    } else {
      MX_QXC(false, false);
    }
#undef MX_QXC
#undef MX_QXP
#undef MX_QX
  };
  bool counted;
  const int rc = LaunchClaiming(ctx, q, n, grid * kWavesPerBlock, stream, noalloc, scratch_base, &counted, launch);
  if (rc != MUONX_OK) return rc;
  MX_HIP(hipGetLastError());
  if (counted) MX_HIP(hipEventRecord(ctx->spill_done, stream));
  return MUONX_OK;
}

// Launches the query kernels for up to kQueryPart rays. With `noalloc` the spill region and the claim
// counters come from the static scratch (the grid is capped so that the spill
// fits), the counters are cleared by a kernel rather than a memset node, no
// stack is in private memory, and no event or buffer is created.
static int LaunchPart(muonx_ctx *ctx, const DevSceneView &s, bool any, bool exact, const QueryArrays &q, uint32_t n,
                      unsigned long long *counters, hipStream_t stream, bool noalloc) {
  TraverseCfg cfg;
  unsigned char *sbase = nullptr;
  int rc;
  if (noalloc) {
    sbase = static_cast<unsigned char *>(StaticScratch(ctx->device));
    if (!sbase) {
      SetError("muonx_intersect_noalloc: no static scratch address for device " + std::to_string(ctx->device));
      return MUONX_ERR_STATE;
    }
  }
  if (exact) return LaunchExactQuery(ctx, s, any, q, n, counters, stream, noalloc, sbase);
  if (noalloc) {
    rc = PlanTraverseShape(ctx->tuning, ctx->num_cus, s.bvh_depth, s.wstack, n, kQueryBlock, cfg, false);
    if (rc != MUONX_OK) return rc;
    if (cfg.gcap > 0) {
      const size_t per_block = size_t(kQueryBlock) * size_t(cfg.gcap) * sizeof(uint2);
      const size_t max_blocks = (kStaticScratchBytes - kStaticScratchHead) / per_block;
      if (max_blocks == 0) {
        SetError("muonx_intersect_noalloc: a traversal stack of " + std::to_string(cfg.kind + cfg.gcap) +
                 " entries per lane needs " + std::to_string(per_block) + " bytes of spill per block, more than the " +
                 std::to_string(kStaticScratchBytes - kStaticScratchHead) + "-byte static scratch");
        return MUONX_ERR_CAPACITY;
      }
      cfg.grid = int(std::min<size_t>(size_t(cfg.grid), max_blocks));
      cfg.threads = cfg.grid * kQueryBlock;
      cfg.spill = reinterpret_cast<uint2 *>(sbase + kStaticScratchHead);
    }
  } else {
    rc = PlanTraverse(ctx, s, n, kQueryBlock, cfg);
    if (rc != MUONX_OK) return rc;
    if ((rc = BeginSpill(ctx, cfg, stream)) != MUONX_OK) return rc;
  }
#define MX_Q(A, C) DispatchTraverse(cfg, QueryLaunch<A, C>{cfg, s, q, n, counters, stream})
  const bool cnt = counters != nullptr;
  const int fetch = ctx->tuning.ray_fetch;
  if (fetch > 0) {  // per-lane ray fetch
    const auto launch = [&](const QueryArrays &q, uint32_t m, uint32_t *next) {
#define MX_QD(A, C) DispatchTraverse(cfg, QueryDynLaunch<A, C>{cfg, s, q, m, counters, next, fetch, stream})
      if (any) {
        if (cnt) MX_QD(true, true);
        else MX_QD(true, false);
      } else {
        if (cnt) MX_QD(false, true);
        else MX_QD(false, false);
      }
#undef MX_QD
    };
    bool counted;
    rc = LaunchClaiming(ctx, q, n, uint32_t(cfg.grid) * kWavesPerBlock, stream, noalloc, sbase, &counted, launch);
    if (rc != MUONX_OK) return rc;
    MX_HIP(hipGetLastError());
    if (counted || (cfg.spill && !noalloc)) MX_HIP(hipEventRecord(ctx->spill_done, stream));
    return MUONX_OK;
  }
  if (any) {
    if (cnt) MX_Q(true, true);
    else MX_Q(true, false);
  } else {
    if (cnt) MX_Q(false, true);
    else MX_Q(false, false);
  }
#undef MX_Q
  MX_HIP(hipGetLastError());
  return noalloc ? MUONX_OK : EndSpill(ctx, cfg, stream);
}

int LaunchQuery(muonx_ctx *ctx, const DevSceneView &s, bool any, bool exact, const float *ro, const float *rd,
                const float *tmax, uint32_t n, int32_t *prim, float *t, uint8_t *occ, unsigned long long *counters,
                hipStream_t stream, bool noalloc) {
  return ForEachPart(QueryArrays{ro, rd, tmax, prim, t, occ}, n, kQueryPart, [&](const QueryArrays &q, uint32_t m) {
    return LaunchPart(ctx, s, any, exact, q, m, counters, stream, noalloc);
  });
}

}  // namespace muonx

using namespace muonx;

namespace {
int CheckQuery(const char *fn, muonx_scene *scene, const muonx_query *q) {
  if (!scene || !q) {
    SetError(std::string(fn) + ": null argument");
    return MUONX_ERR_INVALID;
  }
  if (q->n && (!q->ray_o || !q->ray_d || (q->any_hit ? !q->occluded : !q->prim_id))) {
    SetError(std::string(fn) + ": missing ray or output array");
    return MUONX_ERR_INVALID;
  }
  if (q->mode != MUONX_TRAVERSAL_FAST && q->mode != MUONX_TRAVERSAL_EXACT) {
    SetError(std::string(fn) + ": unknown traversal mode");
    return MUONX_ERR_INVALID;
  }
  return MUONX_OK;
}

int RunQuery(muonx_scene *scene, const muonx_query *q, void *stream, bool noalloc) {
  if (q->mode == MUONX_TRAVERSAL_EXACT && !scene->reference_tree) {
    SetError("exact traversal needs the reference's SAH tree; this scene's BVH was built on the device");
    return MUONX_ERR_STATE;
  }
  std::lock_guard<std::mutex> lock(scene->ctx->mu);
  MX_HIP(hipSetDevice(scene->ctx->device));
  return LaunchQuery(scene->ctx, scene->view, q->any_hit != 0, q->mode == MUONX_TRAVERSAL_EXACT, q->ray_o, q->ray_d,
                     q->tmax, q->n, q->prim_id, q->t, q->occluded, q->counters, static_cast<hipStream_t>(stream),
                     noalloc);
}
}  // namespace

extern "C" int muonx_intersect(muonx_scene *scene, const muonx_query *q, void *stream) {
  const int rc = CheckQuery("muonx_intersect", scene, q);
  return rc != MUONX_OK ? rc : RunQuery(scene, q, stream, false);
}

extern "C" int muonx_intersect_noalloc(muonx_scene *scene, const muonx_query *q, void *stream) {
  const int rc = CheckQuery("muonx_intersect_noalloc", scene, q);
  return rc != MUONX_OK ? rc : RunQuery(scene, q, stream, true);
}

extern "C" int muonx_intersect_closest(muonx_scene *scene, const float *ro, const float *rd, const float *tmax,
                                       uint32_t n, int32_t *prim_id, float *t, void *stream) {
  muonx_query q{ro, rd, tmax, n, 0, MUONX_TRAVERSAL_FAST, prim_id, t, nullptr, nullptr};
  return muonx_intersect(scene, &q, stream);
}

extern "C" int muonx_intersect_any(muonx_scene *scene, const float *ro, const float *rd, const float *tmax,
                                   uint32_t n, uint8_t *occluded, void *stream) {
  muonx_query q{ro, rd, tmax, n, 1, MUONX_TRAVERSAL_FAST, nullptr, nullptr, occluded, nullptr};
  return muonx_intersect(scene, &q, stream);
}
