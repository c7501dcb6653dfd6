// muonx_render: camera ray generation + integrators on the GPU.
// Deterministic integrators (normals / albedo / depth, muon/integration.cc:47-76;
// raytracer / analyticdirect) run as one fused kernel with the exact traversal
// mode (the reference's node visits, so ties and edge hits resolve as in muon);
// the path tracer runs as a wavefront pipeline (pathtracer.hip).
#include <algorithm>
#include <chrono>
#include <climits>
#include <vector>

#include "exact_trace.h"
#include "hitrec.h"
#include "render.h"
#include "wave.h"
#include "rng.h"
#include "runtime.h"

namespace muonx {

void DestroyWorkspace(RenderWorkspace *ws) {
  if (!ws) return;  // the context never rendered
  DestroyContextScheduler(ws);
  if (ws->scratch_busy) (void)hipEventSynchronize(ws->scratch_done);
  if (ws->scratch_done) (void)hipEventDestroy(ws->scratch_done);
  if (ws->ev_in) (void)hipEventDestroy(ws->ev_in);
  if (ws->ev_out) (void)hipEventDestroy(ws->ev_out);
  delete ws;
}

RenderWorkspace *GetWorkspace(muonx_ctx *ctx) {
  if (!ctx->ws) ctx->ws = new RenderWorkspace();
  return ctx->ws;
}

CamParams MakeCam(const muonx_render_params &p) {
  CamParams c;
  c.eye = V3{p.eye[0], p.eye[1], p.eye[2]};
  c.u = V3{p.cam_u[0], p.cam_u[1], p.cam_u[2]};
  c.v = V3{p.cam_v[0], p.cam_v[1], p.cam_v[2]};
  c.w = V3{p.cam_w[0], p.cam_w[1], p.cam_w[2]};
  c.tan_fov_x = p.tan_fov_x;
  c.tan_fov_y = p.tan_fov_y;
  c.width = p.width;
  c.height = p.height;
  return c;
}

// Image kernels: every lane takes one sample of a pixel, follows it to its end
// and takes the next. Samples are handed out in tiles of 8x8 pixels, a
// wavefront's rays being neighbours in both directions; the walks are
// run_walks'. A pixel's samples are added in their order, so the film has the
// reference's bits: with several at once they go to a buffer first
// (k_sum_samples).
struct ImageItems {
  uint32_t width, height, across;
  int first, count;  // the samples of this launch
  uint64_t tile0;    // tile of item 0
  float *buffer;     // count > 1: sample colours, [sample][pixel]
};
struct ImageItem {
  uint32_t px, py, pixel;
  int sample;
};
// Item k: tile k / (64 count), sample, pixel of the tile; false for a pixel
// outside the image (ragged last tiles).
__device__ __forceinline__ bool image_item(const ImageItems &it, uint32_t k, ImageItem &i) {
  const uint32_t wave = k >> 6;
  const uint64_t tile = it.tile0 + wave / uint32_t(it.count);
  i.sample = it.first + int(wave % uint32_t(it.count));
  i.px = uint32_t(tile % it.across) * 8u + (k & 7u);
  i.py = uint32_t(tile / it.across) * 8u + ((k >> 3) & 7u);
  i.pixel = i.py * it.width + i.px;
  return i.px < it.width && i.py < it.height;
}
__device__ __forceinline__ void sample_ray(const CamParams &cam, const ImageItem &i, uint32_t seed, V3 &o, V3 &d) {
  float x, y;
  sample_position(int(i.px), int(i.py), i.sample, path_key(seed, 0, i.pixel, uint32_t(i.sample)), x, y);
  cast_ray(cam, x, y, o, d);
}
// The sample's colour, to the buffer or added to the pixel.
__device__ __forceinline__ void write_sample(const ImageItems &it, const ImageItem &i, V3 c, float *accum) {
  if (it.count > 1) {
    float *out = it.buffer + 3 * (size_t(i.sample - it.first) * it.width * it.height + i.pixel);
    out[0] = c.x;
    out[1] = c.y;
    out[2] = c.z;
  } else {
    float *out = accum + 3 * size_t(i.pixel);
    const V3 acc = i.sample ? V3{out[0], out[1], out[2]} : V3{0.0f, 0.0f, 0.0f};
    out[0] = acc.x + c.x;
    out[1] = acc.y + c.y;
    out[2] = acc.z + c.z;
  }
}
// Adds the buffered samples to the film in their order.
__global__ void k_sum_samples(const float *__restrict__ buffer, int first, int count, uint64_t n,
                              float *__restrict__ accum) {
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) {
    float acc = first ? accum[i] : 0.0f;
    for (int k = 0; k < count; ++k) acc = acc + buffer[uint64_t(k) * n + i];
    accum[i] = acc;
  }
}

// Where this wavefront's counts go.
__device__ __forceinline__ uint32_t CounterSlot() {
  return (blockIdx.x * (kSimpleBlock / 64) + (threadIdx.x >> 6)) % kCounterSlots * kCounterSlotStride;
}
// Idle lanes, beyond those that no sample is left for, at which a wavefront
// stops to give them samples. A tile's rays that start together walk in step:
// at 16, 32 and 64 idle lanes a 1024x1024 depth image of the level-7 icosphere
// takes 672 / 681 / 610 us (12 blocks per CU). Whitted paths differ in length:
// 2202 / 2205 / 3067 us for 500 spheres at 641x479, 4 samples.
constexpr int kSimpleRefill = 64, kWhittedRefill = 16;

// Normals, albedo, depth. Bound by the latency of the few wavefronts along
// silhouettes (lanes 57 % used, 1.1 wavefronts per SIMD on average). Against one
// thread per pixel in rows of 64, a node or a leaf step per iteration, the
// whole stack in LDS and one set of counters: 640x480 normals of the level-6
// icosphere 523 -> 352 us, a 100x100 Cornell box 62 -> 60, 512x512 with four
// samples of 10,000 spheres 1100 -> 441.
template <int CAP>
__global__ void __launch_bounds__(kSimpleBlock) __attribute__((amdgpu_waves_per_eu(4, 8)))
    k_simple(DevSceneView s, CamParams cam, int integrator, int depth0_ok, uint32_t seed, ImageItems it, uint32_t items,
             float *__restrict__ accum, unsigned long long *__restrict__ ctr, uint32_t *next) {
  __shared__ uint2 lds[kPrivateRing * kSimpleBlock];
  uint2 old[PrivateStack<CAP>::kOld];
  PrivateStack<CAP> st(lds + threadIdx.x, kSimpleBlock, old);
  ExactWalk<true, kWalkClosest> w;
  TraceCounters cnt;
  WaveFetch wf(items, kChunk);
  uint32_t traced = 0;
  ImageItem i;
  bool walking = false, have = false, drained = false;
  while (true) {
    const uint64_t needm = __builtin_amdgcn_ballot_w64(!have && !drained);
    if (needm) {
      const uint32_t k = wf.claim(needm, next);
      if (!have && !drained) {
        if (k >= items) {
          drained = true;
        } else if (image_item(it, k, i)) {
          have = true;
          w.hit = -1;
          if (depth0_ok) {
            V3 o, d;
            sample_ray(cam, i, seed, o, d);
            ++traced;
            walking = w.start(s, make_ray(o, d), __builtin_inff(), false, st, cnt);
          }
        }
      }
    }
    const uint64_t drainedm = __builtin_amdgcn_ballot_w64(drained);
    if (__builtin_amdgcn_ballot_w64(have) == 0) {
      if (~drainedm == 0) break;
      continue;
    }
    run_walks(s, w, walking, st, cnt, __popcll(drainedm) + kSimpleRefill);
    if (have && !walking) {
      V3 c{0.0f, 0.0f, 0.0f};
      if (w.hit >= 0) {
        if (integrator == MUONX_INTEGRATOR_ALBEDO) {
          const float *m = s.materials + size_t(s.prim_mat[w.hit]) * kMatStride;
          c = V3{m[3], m[4], m[5]} + V3{m[6], m[7], m[8]};
        } else {
          const HitRecord h = hit_record(s, uint32_t(w.hit), w.r.o, w.r.d);
          if (integrator == MUONX_INTEGRATOR_NORMALS) {
            c = h.normal * 0.5f + 0.5f;
          } else {
            const float z = 1.0f / (1.0f + h.dist);
            c = V3{z, z, z};
          }
        }
      }
      write_sample(it, i, c, accum);
      have = false;
    }
  }
  ctr += CounterSlot();
  wave_count(traced, &ctr[kCtrPrimary]);
  wave_count(cnt.prims, &ctr[kCtrObjectTests]);
  wave_count(cnt.ohits, &ctr[kCtrObjectHits]);
  wave_count(cnt.btests, &ctr[kCtrBoundsTests]);
  wave_count(cnt.bhits, &ctr[kCtrBoundsHits]);
}

// Raytracer (muon/integration.cc:78-120) and AnalyticDirect
// (muon/integration.cc:126-199), deterministic, with the exact traversal
// mode. The raytracer's reflection recursion, color_d = local_d + ks_d *
// color_{d+1}, is evaluated back to front from the stored per-bounce terms so
// that its float operations are the reference's.
constexpr int kWhittedMaxBounces = 32;  // bound for max_depth = -1

// Light::ShadingInfoAt (muon/lighting.cc:7-72); a quad light leaves the
// direction and distance zero, as the reference's restatement does.
__device__ __forceinline__ void shading_info(const float *L, V3 p, V3 &color, V3 &dir, float &dist) {
  const int kind = int(L[0]);
  color = V3{L[1], L[2], L[3]};
  if (kind == MUONX_LIGHT_DIRECTIONAL) {
    dir = V3{L[4], L[5], L[6]};
    dist = __builtin_inff();
  } else if (kind == MUONX_LIGHT_POINT) {
    const V3 to_light = V3{L[4], L[5], L[6]} - p;
    dir = normalize(to_light);
    const float r = length(to_light);
    const float att = L[7] + L[8] * r + L[9] * r * r;
    color = color / att;
    dist = r;
  } else {
    dir = V3{0.0f, 0.0f, 0.0f};
    dist = 0.0f;
  }
}

// A lane goes through its sample's bounces and each bounce's shadow rays as a
// sequence of walks, whichever kind the other lanes are at, so a short path
// waits for no longer one. Bound by instruction issue at 25 % lane use. 500
// shiny spheres under two lights, 641x479, 4 samples, depth 5: 4.08 -> 2.20 ms
// against nested loops in one thread per pixel.
template <int CAP>
__global__ void __launch_bounds__(kSimpleBlock) __attribute__((amdgpu_waves_per_eu(4, 8)))
    k_whitted(DevSceneView s, CamParams cam, int integrator, int cutoff, uint32_t seed, ImageItems it, uint32_t items,
              float *__restrict__ accum, unsigned long long *__restrict__ rays, uint32_t *next) {
  __shared__ uint2 lds[kPrivateRing * kSimpleBlock];
  uint2 old[PrivateStack<CAP>::kOld];
  PrivateStack<CAP> st(lds + threadIdx.x, kSimpleBlock, old);
  ExactWalk<true, kWalkEither> w;
  TraceCounters cnt;
  WaveFetch wf(items, kChunk);
  uint32_t n_primary = 0, n_secondary = 0, n_shadow = 0;
  ImageItem i;
  int nb = 0;  // bounces with a hit (the depth of the next)
  uint32_t light = 0;
  int32_t prim = 0;
  V3 d, color;
  V3 pos, normal;  // the bounce's hit
  V3 local[kWhittedMaxBounces], ks[kWhittedMaxBounces];
  bool walking = false, have = false, drained = false, shadow = false;
  while (true) {
    const uint64_t needm = __builtin_amdgcn_ballot_w64(!have && !drained);
    if (needm) {
      const uint32_t k = wf.claim(needm, next);
      if (!have && !drained) {
        if (k >= items) {
          drained = true;
        } else if (image_item(it, k, i)) {
          have = true;
          nb = 0;
          shadow = false;
          w.hit = -1;
          if (cutoff >= 0) {  // Integrator::Trace returns 0 past the cutoff (muon/integration.cc:29-33)
            V3 o;
            sample_ray(cam, i, seed, o, d);
            ++n_primary;
            walking = w.start(s, make_ray(o, d), __builtin_inff(), false, st, cnt);
          }
        }
      }
    }
    const uint64_t drainedm = __builtin_amdgcn_ballot_w64(drained);
    if (__builtin_amdgcn_ballot_w64(have) == 0) {
      if (~drainedm == 0) break;
      continue;
    }
    run_walks(s, w, walking, st, cnt, __popcll(drainedm) + kWhittedRefill);
    if (have && !walking) {
      bool path_done = false;
      const float *m = s.materials;
      if (!shadow) {
        if (w.hit < 0) {
          path_done = true;
        } else {
          prim = w.hit;
          const HitRecord h = hit_record(s, uint32_t(prim), w.r.o, d);
          pos = h.pos;
          normal = h.normal;
          m += size_t(s.prim_mat[prim]) * kMatStride;
          const V3 amb{m[0], m[1], m[2]}, kd{m[3], m[4], m[5]}, em{m[9], m[10], m[11]};
          if (integrator == MUONX_INTEGRATOR_RAYTRACER) {
            color = amb + em;
            light = 0;
            shadow = true;
          } else {
            color = em;
            for (uint32_t l = 0; l < s.num_lights; ++l) {
              const float *L = s.lights + size_t(l) * kLightStride;
              if (int(L[0]) != MUONX_LIGHT_QUAD) continue;
              const V3 c0{L[4], L[5], L[6]}, e0{L[7], L[8], L[9]}, e1{L[10], L[11], L[12]};
              const V3 verts[4] = {c0, c0 + e0, (c0 + e0) + e1, c0 + e1};
              const V3 brdf = kd * kOneOverPi;
              const V3 radiance{L[1], L[2], L[3]};
              V3 irr{0.0f, 0.0f, 0.0f};
              for (int v = 0; v < 4; ++v) {
                const int ni = (v + 1) % 4;
                const V3 ui = normalize(verts[v] - pos);
                const V3 un = normalize(verts[ni] - pos);
                const float theta = acosf(dot(ui, un));
                const V3 gamma = normalize(cross(ui, un));
                irr = irr + theta * gamma;
              }
              irr = irr * 0.5f;
              color = color + (brdf * radiance) * dot(irr, normal);
            }
            local[nb] = color;
            ks[nb] = V3{0.0f, 0.0f, 0.0f};
            ++nb;
            path_done = true;
          }
        }
      } else {
        m += size_t(s.prim_mat[prim]) * kMatStride;
        if (w.hit < 0) {  // light `light` is visible
          const V3 kd{m[3], m[4], m[5]}, spec{m[6], m[7], m[8]};
          V3 lc, ldir;
          float ldist;
          shading_info(s.lights + size_t(light) * kLightStride, pos, lc, ldir, ldist);
          const V3 diffuse = kd * gmax(dot(normal, ldir), 0.0f);
          const V3 half = normalize(ldir - d);
          const V3 sp = spec * powf(gmax(dot(normal, half), 0.0f), m[12]);
          color = color + lc * (diffuse + sp);
        }
        ++light;
      }
      if (shadow) {
        const V3 shift = pos + kEps * normal;
        if (light < s.num_lights) {
          V3 lc, ldir;
          float ldist;
          shading_info(s.lights + size_t(light) * kLightStride, pos, lc, ldir, ldist);
          ++n_shadow;
          walking = w.start(s, make_ray(shift, ldir), ldist, true, st, cnt);
        } else {
          // the bounce is lit: reflect or end
          const V3 spec{m[6], m[7], m[8]};
          local[nb] = color;
          ks[nb] = spec;
          ++nb;
          shadow = false;
          if ((spec.x > 0.0f || spec.y > 0.0f || spec.z > 0.0f) && nb < kWhittedMaxBounces && nb <= cutoff) {
            d = reflect(d, normal);
            ++n_secondary;
            walking = w.start(s, make_ray(shift, d), __builtin_inff(), false, st, cnt);
          } else {
            path_done = true;
          }
        }
      }
      if (path_done) {
        V3 c{0.0f, 0.0f, 0.0f};
        if (nb > 0) {
          // color_d = local_d + ks_d * color_{d+1}, innermost first; a bounce
          // whose reflected ray found nothing adds ks * 0
          c = local[nb - 1];
          if (ks[nb - 1].x > 0.0f || ks[nb - 1].y > 0.0f || ks[nb - 1].z > 0.0f) c = c + ks[nb - 1] * V3{0.0f, 0.0f, 0.0f};
          for (int b = nb - 2; b >= 0; --b) c = local[b] + ks[b] * c;
        }
        write_sample(it, i, c, accum);
        have = false;
      }
    }
  }
  rays += CounterSlot();
  wave_count(n_primary, &rays[kCtrPrimary]);
  wave_count(n_secondary, &rays[kCtrSecondary]);
  wave_count(n_shadow, &rays[kCtrShadow]);
  wave_count(cnt.prims, &rays[kCtrObjectTests]);
  wave_count(cnt.ohits, &rays[kCtrObjectHits]);
  wave_count(cnt.btests, &rays[kCtrBoundsTests]);
  wave_count(cnt.bhits, &rays[kCtrBoundsHits]);
}

// Blocks per CU of the image kernels. More than their registers let a CU hold
// start late with a chunk of their own, which costs k_whitted (8, 10, 12: 2.20 /
// 2.87 / 2.67 ms above) and helps k_simple's short wavefronts even out (8, 10,
// 12: 668 / 725 / 615 us for the depth image).
constexpr uint32_t kSimpleBlocksPerCu = 12, kWhittedBlocksPerCu = 8;
// The most memory for a launch's samples.
constexpr uint64_t kSampleBytes = uint64_t(64) << 20;

// A render's turn at the workspace's counters and samples, which all renders of
// the context share, on whatever streams they are: its stream waits for the last
// user, and the next user's for it. Held under the context's lock.
class ScratchTurn {
 public:
  ScratchTurn(RenderWorkspace *ws, hipStream_t stream) : ws_(ws), stream_(stream) {}
  ~ScratchTurn() {
    if (!begun_) return;
    // a render that gave up half-way is ordered like any other
    if ((ws_->scratch_done || hipEventCreateWithFlags(&ws_->scratch_done, hipEventDisableTiming) == hipSuccess) &&
        hipEventRecord(ws_->scratch_done, stream_) == hipSuccess) {
      ws_->scratch_busy = true;
    } else {
      (void)hipStreamSynchronize(stream_);
      ws_->scratch_busy = false;
    }
  }
  int Begin() {
    if (ws_->scratch_busy) MX_HIP(hipStreamWaitEvent(stream_, ws_->scratch_done, 0));
    begun_ = true;
    return MUONX_OK;
  }
  // The host has waited for the stream, and so for every user up to this one.
  void Finished() {
    ws_->scratch_busy = false;
    begun_ = false;
  }

 private:
  RenderWorkspace *ws_;
  hipStream_t stream_;
  bool begun_ = false;
};

// Runs one of the deterministic integrators; `counters` holds the trace
// counters and the (cleared) claim counters. Without claim counters the launches
// use no other buffer of the context either: one sample each, added directly, of
// as many pixels as their wavefronts take without.
int RenderDeterministic(muonx_scene *scene, const muonx_render_params &p, float *accum, const RenderCounters &counters,
                        RenderWorkspace *ws, hipStream_t stream) {
  const DevSceneView &s = scene->view;
  if (s.bvh_depth > 96) {
    SetError("BVH too deep for the traversal stack");
    return MUONX_ERR_CAPACITY;
  }
  const CamParams cam = MakeCam(p);
  const uint64_t tiles = ((uint64_t(p.width) + 7) / 8) * ((uint64_t(p.height) + 7) / 8);
  const uint32_t cus = uint32_t(scene->ctx->num_cus > 0 ? scene->ctx->num_cus : 256);
  // samples per launch: their buffer stays within kSampleBytes
  const uint64_t film = uint64_t(p.width) * uint64_t(p.height) * 3 * sizeof(float);
  const int batch =
      counters.claims ? int(std::max<uint64_t>(1, std::min<uint64_t>(uint64_t(p.spp), kSampleBytes / film))) : 1;
  if (batch > 1) {
    const size_t bytes = film * uint64_t(batch);
    if (bytes > ws->samples.bytes && ws->scratch_busy) MX_HIP(hipEventSynchronize(ws->scratch_done));  // it moves
    MX_HIP(ws->samples.Reserve(bytes));
  }
  ImageItems it{uint32_t(p.width), uint32_t(p.height), (uint32_t(p.width) + 7u) >> 3, 0, 0, 0,
                ws->samples.as<float>()};
  unsigned long long *ctr = counters.trace;
  uint32_t *next = counters.claims;
  // muon/integration.cc:29-33
  const int cutoff = p.max_depth == -1 ? INT_MAX : (p.nee != MUONX_NEE_OFF ? p.max_depth - 1 : p.max_depth);
  const bool whitted = p.integrator == MUONX_INTEGRATOR_RAYTRACER || p.integrator == MUONX_INTEGRATOR_ANALYTICDIRECT;
  const uint32_t max_blocks = cus * (whitted ? kWhittedBlocksPerCu : kSimpleBlocksPerCu);
  bool cleared = true;  // the claim counters
  for (it.first = 0; it.first < p.spp; it.first += it.count) {
    it.count = std::min(batch, p.spp - it.first);
    uint64_t part = std::max<uint64_t>(1, (1u << 24) / uint64_t(it.count));  // tiles per launch: below 2^31 items
    if (!next) part = std::min(part, UnclaimedItems(max_blocks * (kSimpleBlock / 64)) / 64);
    for (it.tile0 = 0; it.tile0 < tiles; it.tile0 += part) {
      const uint32_t items = uint32_t(std::min(tiles - it.tile0, part)) * uint32_t(it.count) * 64u;
      const uint32_t blocks = ClaimBlocks(items, max_blocks, kSimpleBlock / 64);
      if (NeedsClaims(items, blocks * (kSimpleBlock / 64))) {
        if (!cleared) MX_HIP(hipMemsetAsync(next, 0, kClaimBytes, stream));
        cleared = false;
      }
      const dim3 grid(blocks), block(kSimpleBlock);
#define MX_IMAGE(CAP)                                                                                                \
  if (whitted)                                                                                                       \
    hipLaunchKernelGGL(k_whitted<CAP>, grid, block, 0, stream, s, cam, p.integrator, cutoff, p.seed, it, items, accum, \
                       ctr, next);                                                                                   \
  else                                                                                                               \
    hipLaunchKernelGGL(k_simple<CAP>, grid, block, 0, stream, s, cam, p.integrator, cutoff >= 0 ? 1 : 0, p.seed, it,  \
                       items, accum, ctr, next)
      if (s.bvh_depth <= 24) {
        MX_IMAGE(24);
      } else if (s.bvh_depth <= 48) {
        MX_IMAGE(48);
      } else {
        MX_IMAGE(96);
      }
#undef MX_IMAGE
    }
    if (it.count > 1) {
      const uint64_t n = film / sizeof(float);
      hipLaunchKernelGGL(k_sum_samples, dim3(uint32_t(std::min<uint64_t>(4096, (n + 255) / 256))), dim3(256), 0, stream,
                         it.buffer, it.first, it.count, n, accum);
    }
  }
  MX_HIP(hipGetLastError());
  return MUONX_OK;
}

}  // namespace muonx

using namespace muonx;

namespace {
// muonx_render with the context's lock held.
int RenderLocked(muonx_scene *scene, const muonx_render_params &p, float *accum, muonx_trace_stats *stats,
                 hipStream_t stream) {
  if (p.width <= 0 || p.height <= 0 || p.spp <= 0) {
    SetError("muonx_render: width, height and spp must be positive");
    return MUONX_ERR_INVALID;
  }
  if (!p.has_camera) {
    SetError("muonx_render: scene has no camera");  // the reference dereferences a null camera
    return MUONX_ERR_INVALID;
  }
  if (p.integrator != MUONX_INTEGRATOR_PATHTRACER && !scene->reference_tree) {
    SetError("muonx_render: this integrator traverses the reference's SAH tree; the scene's BVH was built on "
             "the device");
    return MUONX_ERR_STATE;
  }
  muonx_ctx *ctx = scene->ctx;
  MX_HIP(hipSetDevice(ctx->device));
  bool capturing = false;
  int rc = IsCapturing(stream, &capturing);
  if (rc != MUONX_OK) return rc;
  if (capturing && p.integrator == MUONX_INTEGRATOR_PATHTRACER) {
    // the host polls the engine's counters: nothing may reach its stream, whose work the graph would take in
    SetError("muonx_render: the path tracer cannot be captured into a graph");
    return MUONX_ERR_STATE;
  }
  RenderWorkspace *ws = GetWorkspace(ctx);
  MX_HIP(ws->counters.Reserve(kRenderCounterBytes + kTraceCounterBytes));  // allocated once, never moved
  ScratchTurn turn(ws, stream);
  if (p.integrator != MUONX_INTEGRATOR_PATHTRACER && !capturing) {
    if ((rc = turn.Begin()) != MUONX_OK) return rc;
    MX_HIP(hipMemsetAsync(ws->counters.ptr, 0, kRenderCounterBytes, stream));
  }
  hipEvent_t e0, e1;
  MX_HIP(hipEventCreate(&e0));
  MX_HIP(hipEventCreate(&e1));
  MX_HIP(hipEventRecord(e0, stream));
  const size_t trace_at = capturing ? kRenderCounterBytes : kClaimBytes;
  const RenderCounters ctr{ws->counters.as<unsigned long long>() + trace_at / sizeof(unsigned long long),
                           capturing ? nullptr : ws->counters.as<uint32_t>()};
  bool host_rays = false;
  unsigned long long rays[kEngineCounters] = {};
  switch (p.integrator) {
    case MUONX_INTEGRATOR_NORMALS:
    case MUONX_INTEGRATOR_ALBEDO:
    case MUONX_INTEGRATOR_DEPTH:
    case MUONX_INTEGRATOR_RAYTRACER:
    case MUONX_INTEGRATOR_ANALYTICDIRECT:
      rc = RenderDeterministic(scene, p, accum, ctr, ws, stream);
      break;
    case MUONX_INTEGRATOR_PATHTRACER:
      rc = RenderPathTracer(scene, p, accum, stream, rays);
      host_rays = true;
      break;
    default:
      SetError("muonx_render: integrator " + std::to_string(p.integrator) + " is not on the GPU render path");
      rc = MUONX_ERR_INVALID;
  }
  if (rc != MUONX_OK) {
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
  }
  MX_HIP(hipEventRecord(e1, stream));
  if (stats) {
    unsigned long long h[kNumCounters] = {};
    if (!host_rays) {
      std::vector<unsigned long long> slots(kTraceCounterBytes / sizeof(unsigned long long));
      MX_HIP(hipMemcpyAsync(slots.data(), ctr.trace, kTraceCounterBytes, hipMemcpyDeviceToHost, stream));
      MX_HIP(hipStreamSynchronize(stream));
      for (uint32_t k = 0; k < kCounterSlots; ++k)
        for (int c = 0; c < kNumCounters; ++c) h[c] += slots[size_t(k) * kCounterSlotStride + size_t(c)];
    }
    MX_HIP(hipStreamSynchronize(stream));
    if (!host_rays) turn.Finished();
    float ms = 0.0f;
    MX_HIP(hipEventElapsedTime(&ms, e0, e1));
    stats->primary_rays = host_rays ? rays[0] : h[kCtrPrimary];
    stats->secondary_rays = host_rays ? rays[1] : h[kCtrSecondary];
    stats->shadow_rays = host_rays ? rays[2] : h[kCtrShadow];
    stats->render_ns = uint64_t(double(ms) * 1e6);
    stats->culled_rays = host_rays ? rays[3] : 0;
    // the path tracer's: the work of its traversals in the device tree
    stats->object_tests = host_rays ? rays[4] : h[kCtrObjectTests];
    stats->object_hits = host_rays ? rays[5] : h[kCtrObjectHits];
    stats->bounds_tests = host_rays ? rays[6] : h[kCtrBoundsTests];
    stats->bounds_hits = host_rays ? rays[7] : h[kCtrBoundsHits];
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return MUONX_OK;
}
}  // namespace

extern "C" int muonx_render(muonx_scene *scene, const muonx_render_params *params, float *accum,
                            muonx_trace_stats *stats, void *stream) {
  if (!scene || !params || !accum) {
    SetError("muonx_render: null argument");
    return MUONX_ERR_INVALID;
  }
  std::lock_guard<std::mutex> lock(scene->ctx->mu);
  return RenderLocked(scene, *params, accum, stats, static_cast<hipStream_t>(stream));
}

extern "C" int muonx_render_host(muonx_scene *scene, const muonx_render_params *params, float *accum_host,
                                 muonx_trace_stats *stats) {
  if (!scene || !params || !accum_host) {
    SetError("muonx_render_host: null argument");
    return MUONX_ERR_INVALID;
  }
  if (params->width <= 0 || params->height <= 0) {
    SetError("muonx_render_host: width and height must be positive");
    return MUONX_ERR_INVALID;
  }
  const size_t bytes = size_t(params->width) * size_t(params->height) * 3 * sizeof(float);
  // one call at a time from the film's allocation to its copy: the next may move it
  std::lock_guard<std::mutex> lock(scene->ctx->mu);
  MX_HIP(hipSetDevice(scene->ctx->device));
  RenderWorkspace *ws = GetWorkspace(scene->ctx);
  MX_HIP(ws->film.Reserve(bytes));
  float *dev = ws->film.as<float>();
  const int rc = RenderLocked(scene, *params, dev, stats, nullptr);
  if (rc != MUONX_OK) return rc;
  MX_HIP(hipMemcpy(accum_host, dev, bytes, hipMemcpyDeviceToHost));
  return MUONX_OK;
}
