// The exact traversal (the reference's node visits, box_hit_exact) as
// resumable walks of a wavefront's lanes: what the exact queries and the
// deterministic integrators run.
#ifndef MUONX_DEVICE_EXACT_TRACE_H_
#define MUONX_DEVICE_EXACT_TRACE_H_

#include "trace.h"

namespace muonx {

// Which queries a walk answers: Intersect, HasIntersection, or either, as
// start() is told.
constexpr int kWalkClosest = 0, kWalkAny = 1, kWalkEither = 2;

// One lane's walk. COUNT counts the reference's tests (TraceCounters). It
// holds at most the binary tree's depth minus one stack entries.
template <bool COUNT, int KIND>
struct ExactWalk {
  TraceRay r;
  float best;
  int32_t hit;   // leaf-order primitive or -1
  uint32_t ref;  // the node or leaf to visit next
  ObjCache oc;
  bool plain, any_hit;
  uint32_t missed;  // counting any-hit walks: missed far children not popped yet

  __device__ __forceinline__ bool any() const { return KIND == kWalkEither ? any_hit : KIND == kWalkAny; }
  __device__ __forceinline__ bool at_leaf() const { return (ref & kLeafBit) != 0u; }
  // Linear::HasIntersection counts nothing (muon/acceleration.cc:33-45).
  __device__ __forceinline__ bool counts(const DevSceneView &s) const { return COUNT && !(s.linear && any()); }

  // False when the walk is over at once (counting: the ray misses the root's box).
  template <class Stack>
  __device__ __forceinline__ bool start(const DevSceneView &s, const TraceRay &ray, float tmax, bool any_query,
                                        Stack &st, TraceCounters &cnt) {
    r = ray;
    best = tmax;
    hit = -1;
    ref = 0;
    oc.tid = -1;
    any_hit = any_query;
    missed = 0;
    plain = plain_ray(s, ray);
    st.reset();
    if (!counts(s)) return true;
    const float4 *np = s.nodes;
    if (s.linear) {
      // Linear::Intersect tests every primitive and no bounds
      // (muon/acceleration.cc:14-31): the one leaf is node 0's first child
      ref = __float_as_uint(ldg(np + 3).x);
      return true;
    }
    // The reference tests the root's box first (muon/acceleration.cc:92-99);
    // here it is the union of node 0's child boxes. A ray that misses it
    // misses every box below, so stopping changes no result. A root that is
    // a leaf sits in node 0's first child (the second is a sentinel).
    const float4 n0 = ldg(np), n1 = ldg(np + 1), n2 = ldg(np + 2);
    float lo;
    cnt.btests++;
    if (!box_hit_exact(r, plain, fminf(n0.x, n1.x), fmaxf(n0.y, n1.y), fminf(n0.z, n1.z), fmaxf(n0.w, n1.w),
                       fminf(n2.x, n2.z), fmaxf(n2.y, n2.w), best, lo))
      return false;
    cnt.bhits++;
    if (s.root_leaf) ref = __float_as_uint(ldg(np + 3).x);
    return true;
  }

  // The next stack entry whose box starts before `best`; false when there is
  // none. Counting, a popped far child is the reference's bounds test at its
  // pop.
  template <class Stack>
  __device__ __forceinline__ bool pop(const DevSceneView &s, Stack &st, TraceCounters &cnt) {
    const bool count = counts(s);
    while (!st.empty()) {
      const uint2 e = st.pop();
      if (count) cnt.btests++;
      // (an any-hit walk's `best` stays its tmax, which the box passed when
      // it was pushed)
      if (any() || __uint_as_float(e.y) < best) {
        if (count) cnt.bhits++;
        if (any()) missed = e.y;
        ref = e.x;
        return true;
      }
    }
    return false;
  }

  // Visits the internal node `ref`, near child (reference order:
  // children[dir[axis] < 0], muon/acceleration.cc:134-138) first; false when
  // the walk is over.
  template <class Stack>
  __device__ __forceinline__ bool node(const DevSceneView &s, Stack &st, TraceCounters &cnt) {
    const float4 *np = s.nodes + 4 * size_t(ref);
    const float4 n0 = ldg(np), n1 = ldg(np + 1), n2 = ldg(np + 2);
    const int4 n3 = ldg(reinterpret_cast<const int4 *>(np + 3));
    const bool count = counts(s);
    if (COUNT) cnt.nodes++;
    float lo0, lo1;
    const bool h0 = box_hit_exact(r, plain, n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, best, lo0);
    const bool h1 = box_hit_exact(r, plain, n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, best, lo1);
    const uint32_t axis = (uint32_t(n3.z) >> 29) & 3u;
    const bool swap = (r.dneg >> axis) & 1u;  // near child is children[1]
    const uint32_t near_ref = swap ? uint32_t(n3.y) : uint32_t(n3.x);
    const uint32_t far_ref = swap ? uint32_t(n3.x) : uint32_t(n3.y);
    const bool hn = swap ? h1 : h0;
    const bool hf = swap ? h0 : h1;
    const float lof = swap ? lo0 : lo1;
    if (count) {
      // The reference (muon/acceleration.cc:137,197) always pushes the far
      // child and tests its box only when it pops it, which an any-hit query
      // that stops at its first hit (:182-183) may never do. A far child
      // whose box is missed would be popped for that test alone, so it is
      // counted here and not pushed; an any-hit walk takes back the tests of
      // those it did not come to (`missed`, as it was when the entry it works
      // on was pushed, plus those met since). With the near box missed the
      // far one is popped at once.
      cnt.btests += hn && hf ? 1u : 2u;
      cnt.bhits += uint32_t(hn || hf);
      missed += uint32_t(hn && !hf);
    }
    if (hn) {
      if (hf) st.push(make_uint2(far_ref, any() ? missed : __float_as_uint(lof)));
      ref = near_ref;
      return true;
    }
    if (hf) {
      ref = far_ref;
      return true;
    }
    return pop(s, st, cnt);
  }

  // Tests the primitives of the leaf `ref`; false when the walk is over.
  template <class Stack>
  __device__ __forceinline__ bool leaf(const DevSceneView &s, Stack &st, TraceCounters &cnt) {
    const bool count = counts(s);
    for (uint32_t i = ref & ~kLeafBit;; ++i) {
      float dist;
      uint32_t flags;
      const bool ph = prim_hit(s, i, r, oc, dist, flags);
      const bool closer = ph && dist > 0.0f && dist < best;
      if (count) {
        cnt.prims++;
        // an object hit is Primitive::Intersect's (closest hit) or
        // HasIntersection's (any hit: also 0 < dist < tmax), muon/objects.cc:9-17
        if (any() ? closer : ph) cnt.ohits++;
      }
      if (closer) {
        best = dist;
        hit = int32_t(i);
        if (any()) {
          if (count) cnt.btests -= missed;
          return false;
        }
      }
      if (flags & 1u) break;
    }
    return pop(s, st, cnt);
  }
};

}  // namespace muonx

#endif
