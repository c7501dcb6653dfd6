// Launch-side selection of the traversal variant (stack policy, loop form)
// from a context's tuning, shared by the query and path-tracer kernels.
#ifndef MUONX_DEVICE_TRAVERSE_LAUNCH_H_
#define MUONX_DEVICE_TRAVERSE_LAUNCH_H_

#include <algorithm>

#include "runtime.h"
#include "trace.h"
#include "wave.h"

namespace muonx {

// Stack variants: kinds 24/48/96 = full LDS stack of that capacity, 8 = LDS
// ring of 8 with older entries in private memory (kPrivateCap in all), 16 =
// LDS ring of 16 with HBM spill.
constexpr int kPrivateCap = 72;
struct TraverseCfg {
  int kind;     // 24, 48, 96, 8 or 16
  bool ww;
  int width;    // node format: kNodesBinary, kNodesWide, kNodesWideQ
  int grid;     // persistent blocks
  int threads;  // grid * block
  uint2 *spill;
  int gcap;     // spill entries per thread
};

// Everything a kernel needs to build its stack.
struct StackArgs {
  uint2 *spill;
  int gcap;
};

template <int KIND>
struct StackOf;
template <>
struct StackOf<24> { using T = LdsStack<24>; static constexpr int kLds = 24, kPrivate = 1; };
template <>
struct StackOf<48> { using T = LdsStack<48>; static constexpr int kLds = 48, kPrivate = 1; };
template <>
struct StackOf<96> { using T = LdsStack<96>; static constexpr int kLds = 96, kPrivate = 1; };
template <>
struct StackOf<8> {
  using T = PrivateStack<kPrivateCap>;
  static constexpr int kLds = kPrivateRing, kPrivate = T::kOld;
};
template <>
struct StackOf<16> { using T = RingStack<16>; static constexpr int kLds = 16, kPrivate = 1; };

// `old`: a kernel's private array of StackOf<KIND>::kPrivate entries.
template <int KIND>
__device__ __forceinline__ typename StackOf<KIND>::T make_stack(uint2 *lds, int block, const StackArgs &sa,
                                                                uint2 *old) {
  if constexpr (KIND == 8) {
    return typename StackOf<KIND>::T(lds + threadIdx.x, block, old);
  } else if constexpr (KIND == 16) {
    const int gtid = int(blockIdx.x) * block + int(threadIdx.x);
    const int nthreads = int(gridDim.x) * block;
    return typename StackOf<KIND>::T(lds + threadIdx.x, block, sa.spill + gtid, nthreads, sa.gcap);
  } else {
    return typename StackOf<KIND>::T(lds + threadIdx.x, block);
  }
}

// Resolves the variant for a scene (binary depth, wide-stack bound): node
// format, grid, stack kind and the spill entries per thread (cfg.gcap; the
// spill region then needs cfg.threads * cfg.gcap uint2, not yet assigned).
// Without `private_stacks` no kind is chosen whose stack lives in private
// memory, which the runtime provides for every resident wavefront of the card
// at a kernel's first dispatch (264 MiB for kind 8). Allocates nothing.
inline int PlanTraverseShape(const muonx_tuning &t, int num_cus, uint32_t bvh_depth, uint32_t wstack,
                             uint64_t work_items, int block, TraverseCfg &cfg, bool private_stacks = true) {
  const int cus = num_cus > 0 ? num_cus : 256;
  cfg.width = t.bvh_width != 4 ? kNodesBinary : (t.node_bits == 8 ? kNodesWideQ : kNodesWide);
  const int bpc = std::max(1, t.blocks_per_cu);
  cfg.grid = int(ClaimBlocks(work_items, uint32_t(cus * bpc), uint32_t(block / 64)));
  cfg.threads = cfg.grid * block;
  cfg.ww = t.while_while != 0;
  cfg.spill = nullptr;
  cfg.gcap = 0;
  // binary: entries never exceed depth - 1; wide: the collapse's bound
  const int need = int(cfg.width != kNodesBinary ? std::max<uint32_t>(wstack, 1) : bvh_depth);
  const bool ring = t.stack_entries == 8 || t.stack_entries == 16;
  if (ring && private_stacks && need <= (t.stack_entries == 8 ? kPrivateCap : 8)) {
    cfg.kind = 8;
    return MUONX_OK;
  }
  if (ring || need > 96) {
    cfg.kind = 16;
    cfg.gcap = std::max(0, need - 16);
    return MUONX_OK;
  }
  if (need <= 24) cfg.kind = 24;
  else if (need <= 48) cfg.kind = 48;
  else cfg.kind = 96;
  return MUONX_OK;
}

// PlanTraverseShape, then reserves the spill region in `spill`.
inline int PlanTraverseInto(const muonx_tuning &t, int num_cus, uint32_t bvh_depth, uint32_t wstack,
                            uint64_t work_items, int block, DevBuf &spill, TraverseCfg &cfg) {
  const int rc = PlanTraverseShape(t, num_cus, bvh_depth, wstack, work_items, block, cfg);
  if (rc != MUONX_OK || cfg.gcap == 0) return rc;
  MX_HIP(spill.Reserve(size_t(cfg.threads) * cfg.gcap * sizeof(uint2)));
  cfg.spill = spill.as<uint2>();
  return MUONX_OK;
}

inline int PlanTraverse(muonx_ctx *ctx, const DevSceneView &s, uint64_t work_items, int block, TraverseCfg &cfg) {
  return PlanTraverseInto(ctx->tuning, ctx->num_cus, s.bvh_depth, s.wstack, work_items, block, ctx->spill, cfg);
}

// Kernels that use the spill region wait for its previous user when issued
// on another stream.
inline int BeginSpill(muonx_ctx *ctx, const TraverseCfg &cfg, hipStream_t stream) {
  if (!cfg.spill) return MUONX_OK;
  if (!ctx->spill_done) MX_HIP(hipEventCreateWithFlags(&ctx->spill_done, hipEventDisableTiming));
  MX_HIP(hipStreamWaitEvent(stream, ctx->spill_done, 0));
  return MUONX_OK;
}
inline int EndSpill(muonx_ctx *ctx, const TraverseCfg &cfg, hipStream_t stream) {
  if (!cfg.spill) return MUONX_OK;
  MX_HIP(hipEventRecord(ctx->spill_done, stream));
  return MUONX_OK;
}

// Calls F::template run<KIND, WW, WIDTH>() for the planned variant.
template <int W, class F>
inline void DispatchKind(const TraverseCfg &cfg, F &&f) {
  switch (cfg.kind) {
    case 8: cfg.ww ? f.template run<8, true, W>() : f.template run<8, false, W>(); break;
    case 16: cfg.ww ? f.template run<16, true, W>() : f.template run<16, false, W>(); break;
    case 24: cfg.ww ? f.template run<24, true, W>() : f.template run<24, false, W>(); break;
    case 48: cfg.ww ? f.template run<48, true, W>() : f.template run<48, false, W>(); break;
    default: cfg.ww ? f.template run<96, true, W>() : f.template run<96, false, W>(); break;
  }
}
template <class F>
inline void DispatchTraverse(const TraverseCfg &cfg, F &&f) {
  if (cfg.width == kNodesWideQ) DispatchKind<kNodesWideQ>(cfg, f);
  else if (cfg.width == kNodesWide) DispatchKind<kNodesWide>(cfg, f);
  else DispatchKind<kNodesBinary>(cfg, f);
}
}  // namespace muonx

#endif
