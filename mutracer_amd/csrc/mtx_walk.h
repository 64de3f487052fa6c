// Wave-scheduled two-level traversal: the inner loop of the ray-query and
// wavefront trace kernels.
//
// Each lane walks its ray exactly as traverse() (mtx_accel.h) does: the same
// nodes in the same order, the same box and triangle arithmetic and the same
// hit-update rule, so its hit is bit-identical. What differs is when a lane's
// next piece of work runs. A lane is at an interior node (of either level), at
// a triangle of a BLAS leaf, or between instances (a TLAS leaf, the end of a
// BLAS). Run in lockstep, a wave whose lanes are spread over these executes
// all three bodies per iteration with a few lanes each (22% of the lanes of an
// instruction were active). Here the wave counts its lanes, runs the body that
// most of them wait for and lets the others wait, and takes new rays for the
// lanes that have finished once enough of them have (36% active).
//
// What bounds it (1M-triangle 1080p step, closest hit): the vector memory
// address unit is busy 77% of the cycles (about 27 cycles per 16-byte load of
// a wave, whatever its active lanes) and the VALU issues 62% of them, both in
// proportion to the waves' iterations. 82 -> 50 ms for its 80M closest-hit
// rays, 49 -> 26 ms for its 51M shadow rays (in kernels of their own); 4096
// rays in a 50k-triangle mesh 250 -> 104 us. Rays that share nothing are bound
// by the caches' misses instead: 4M scattered rays in 1M triangles miss the L2
// with 62% of their requests, some 66 GB in 9.1 ms. Fetching each node by the
// four lanes of a quad (16 bytes each, through LDS) quarters the cache accesses
// but not the address unit's time and measured slower (56-59 ms), as did
// returning to the TLAS within the node step (53 ms: fewer waits, more
// instructions in every step).
#pragma once
#include "mtx_accel.h"
#include "mtx_fetch.h"

namespace mtx {

// A wave keeps to interior nodes while at least kBoxEighths / 8 of its active
// lanes are at one: 2, 3 and 4 measure 52.3, 50.8 and 50.8 ms for closest hit
// and 27.1, 26.1 and 26.4 ms for shadow rays at the 1M-triangle 1080p step
// (each in a kernel of its own).
constexpr int kBoxEighths = 3;

// What a lane traces: filled by the kernel's load(i, ray).
struct RayIn {
  f3 o, d;
  float tMax;
  int32_t curTri, curSlot;  // the triangle this ray must skip (curSlot -1: none)
  const AccelView *acc;     // kMulti: the ray's scene
  uint32_t id;              // handed to covers() and done()
};
// Traces queue entries 0 .. n-1, each once: load(i, RayIn&) reads entry i,
// hit(id, t, barycentrics, slot, tri, source) takes each accepted triangle of
// a closest-hit query (the last one given is the closest), covers(id, slot,
// tri, barycentrics) is the coverage test of masked instances (any hit), and
// done(id, any, counters) ends the entry. `ctr` is the queue's chunk counters
// (none with kStatic) and kReverse its order of waves (WorkQueue).
template <bool kAnyHit, bool kCount, bool kMulti, bool kMasked, bool kReverse, bool kStatic, class Stack, class Load, class Hit, class Covers, class Done>
__device__ __forceinline__ void trace_queue(uint32_t n, uint32_t *ctr, const AccelView &one, bool doubleSided, Stack &st,
                                            Load &&load, Hit &&hit, Covers &&covers, Done &&done) {
  // cur >= 0: the interior node to visit; cur < kIdle: a leaf (of the BLAS
  // while inBlas, else of the TLAS); kReturn: the current subtree is done.
  constexpr int32_t kReturn = -1, kIdle = -2;
  WorkQueue<kStatic> wq(n, ctr, kReverse);
  const uint32_t lane = lane_id();
  uint32_t id = 0;
  f3 ro = splat(0.0f), rd = ro, winv = ro, o = ro, invD = ro, shear = ro;
  float tMax = 0.0f;
  int32_t cur = kIdle, sp = 0, base = 0, leafRemaining = 0, triLeft = 0;
  int32_t slotIdx = -1, curTri = -1, curSlot = -1;
  int maxDim = 2;
  bool inBlas = false, cull = false, masked = false, any = false, live = false;
  const MTX_AS_GLOBAL TNode *nodes = nullptr;
  const MTX_AS_GLOBAL TriRec *btris = nullptr;
  const MTX_AS_GLOBAL TNode *tnodes = as_global(one.tlasNodes);
  const MTX_AS_GLOBAL InstSlot *slots = as_global(one.slots);
  bool perInst = one.perInstanceBounds != 0u;
  TraceCounters cnt{0u, 0u, 0u};

  while (true) {
    const uint64_t mIdle = __ballot(cur == kIdle) & wq.laneMask;
    const int nIdle = __popcll(mIdle);
    if (nIdle >= wq.refillMin && wq.more()) {
      // Results out and new rays in, for all lanes that wait for them at once.
      uint32_t first;
      const uint32_t take = wq.take((uint32_t)nIdle, first);
      const uint32_t rank = (uint32_t)__popcll(mIdle & ((1ull << lane) - 1ull));
      if (cur == kIdle && live) {
        done(id, any, cnt);
        live = false;
      }
      if (((mIdle >> lane) & 1ull) && rank < take) {
        RayIn r;
        load(first + rank, r);
        live = true;
        id = r.id;
        ro = r.o;
        rd = r.d;
        tMax = r.tMax;
        curTri = r.curTri;
        curSlot = r.curSlot;
        any = false;
        if (kCount) cnt = TraceCounters{0u, 0u, 0u};
        winv = splat(1.0f) / rd;
        o = ro;
        invD = winv;
        sp = 0;
        base = 0;
        leafRemaining = 0;
        triLeft = 0;
        inBlas = false;
        const AccelView &av = kMulti ? *r.acc : one;
        if (kMulti) {
          tnodes = as_global(av.tlasNodes);
          slots = as_global(av.slots);
          perInst = av.perInstanceBounds != 0u;
        }
        nodes = tnodes;
        if (av.empty == 0u) {
          if (kCount) cnt.boxes++;
          if (intersect_box(o, f3{av.rootMin[0], av.rootMin[1], av.rootMin[2]},
                            f3{av.rootMax[0], av.rootMax[1], av.rootMax[2]}, invD, tMax) > 0.0f)
            cur = av.tlasRootRef;
        }
      }
      continue;
    }
    const int nAct = wq.lanes - nIdle;
    if (nAct == 0) break;
    const int boxMin = max(1, (nAct * kBoxEighths) >> 3);
    int nBox = __popcll(__ballot(cur >= 0));
    const int nTri = __popcll(__ballot(inBlas && cur < kIdle)), nInst = nAct - nBox - nTri;
    if (nBox >= boxMin || nBox >= max(nTri, nInst)) {
      do {
        if (cur >= 0) {
          const TNode nd = nodes[cur];
          const float d0 = intersect_box(o, f3of(nd.a), f3of(nd.b), invD, tMax);
          const float d1 = intersect_box(o, f3of(nd.c), f3of(nd.d), invD, tMax);
          if (kCount) cnt.boxes += 2;
          const int32_t left = fint(nd.a.w), right = fint(nd.b.w);
          const bool rightNear = d0 > d1;
          const int32_t nearRef = rightNear ? right : left, farRef = rightNear ? left : right;
          const float dn = rightNear ? d1 : d0, df = rightNear ? d0 : d1;
          const bool nearHit = dn > 0.0f, farHit = df > 0.0f;
          cur = nearHit ? nearRef : farRef;
          if (nearHit) {
            if (farHit) st.put(sp++, farRef);
          } else if (!farHit) {
            cur = kReturn;
            if (sp > base) cur = st.get(--sp);
          }
        }
        nBox = __popcll(__ballot(cur >= 0));
      } while (nBox >= boxMin);
    } else if (nTri >= nInst) {
      if (inBlas && cur < kIdle) {
        const int32_t tri = cur & 0x7fffffff;
        const TriRec r = btris[tri];
        if (triLeft == 0) triLeft = fint(r.v1.w);
        if (triLeft > 0 && !(tri == curTri && slotIdx == curSlot)) {
          const f3 p0 = f3of(r.v0), p1 = f3of(r.v1), p2 = f3of(r.v2);
          if (kCount) cnt.tris++;
          f3 b;
          const float tt = intersect_triangle(o, p0, p1, p2, maxDim, shear, tMax, b);
          if (tt > 0.0f) {
            bool take = true;
            if (!kAnyHit && cull) {  // the instance-space direction, computed again as on entry
              const MTX_AS_GLOBAL InstSlot &s = slots[slotIdx];
              const float4 c0 = s.c0, c1 = s.c1, c2 = s.c2, c3 = s.c3;
              const f3 d = xform(Affine{f3of(c0), f3of(c1), f3of(c2), f3of(c3)}, rd, 0.0f);
              take = !(dot(normalize(cross(p1 - p0, p2 - p0)), d) > 0.0f);
            }
            if (kMasked && take && masked) take = covers(id, slotIdx, tri, b);
            if (take) {
              any = true;
              if (!kAnyHit) {
                tMax = tt;
                hit(id, tt, b, slotIdx, tri, fint(r.v0.w));
              }
            }
          }
        }
        cur++;
        triLeft--;
        if (triLeft <= 0) {
          triLeft = 0;
          cur = kReturn;
          if (sp > base) cur = st.get(--sp);
        }
        if (kAnyHit && any) cur = kIdle;
      }
    } else {
      if (cur < 0 && cur != kIdle && !(inBlas && cur < kIdle)) {
        if (inBlas) {  // back to the world ray
          inBlas = false;
          base = 0;
          o = ro;
          invD = winv;
          nodes = tnodes;
        }
        if (cur == kReturn && leafRemaining <= 0) cur = sp > 0 ? st.get(--sp) : kIdle;
        if (cur < 0 && cur != kIdle) {
          if (cur != kReturn) {
            slotIdx = cur & 0x7fffffff;
            leafRemaining = fint(slots[slotIdx].c1.w);
            slotIdx += leafRemaining;  // last instance first
          }
          cur = kReturn;
          leafRemaining--;
          slotIdx--;
          bool enter = leafRemaining >= 0;
          if (enter) {
            const MTX_AS_GLOBAL InstSlot &s = slots[slotIdx];
            if (perInst) {
              if (kCount) cnt.boxes++;
              enter = intersect_box(ro, f3of(s.bmin), f3of(s.bmax), winv, tMax) > 0.0f;
            }
            if (enter) {
              if (kCount) cnt.instances++;
              const float4 c0 = s.c0, c1 = s.c1, c2 = s.c2, c3 = s.c3;
              const Affine w2l{f3of(c0), f3of(c1), f3of(c2), f3of(c3)};
              o = xform(w2l, ro, 1.0f);
              const f3 d = xform(w2l, rd, 0.0f);
              invD = splat(1.0f) / d;
              maxDim = max_dimension(vabs(d));
              shear = get_shear(d, invD, maxDim);
              if (!kAnyHit) cull = !doubleSided && (fbits(c3.w) & 1u) == 0u;
              if (kMasked) masked = (fbits(c3.w) & kSlotMasked) != 0u;
              nodes = as_global(s.nodes);
              btris = as_global(s.tris);
              inBlas = true;
              base = sp;
              cur = fint(c0.w);
            }
          }
        }
      }
    }
  }
  if (live) done(id, any, cnt);
}

}  // namespace mtx
