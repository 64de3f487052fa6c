// Work distribution and occupancy targets of the traversal kernels (gfx950:
// 64-lane waves, 8 XCDs each with its own L2).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mtx_split.h"

namespace mtx {

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }

// Ordering point for LDS between the lanes of one wave: what they stored
// before it, the others load after it. (The barrier alone orders nothing in
// memory, it only keeps the instructions together.)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kXcds = 8;

// Occupancy the register allocator must reach for the traversal kernels
// (waves per SIMD): 5 (96 VGPRs) for the wavefront kernels and closest-hit
// queries, where 6 spills (closest hit of the 1M-triangle 1080p step 66.5 ms
// against 50.2, 4 waves 62 ms; shadow rays 26.1 against 25.8; each in a kernel
// of its own), 6 (no spill) for the smaller any-hit query (1.01 ms against 1.04
// for 1.5M rays).
constexpr int kTraceWaves = 5;
constexpr int kOcclusionWaves = 6;

// Idle lanes a wave gathers before it takes new rays: loading a ray and
// writing a result cost about a hundred instructions whatever the number of
// lanes. 8, 16 and 24 measure within 1%.
constexpr int kRefill = 16;

// Words between the chunk counters of two XCDs: each counter on lines of its
// own, so that an atomic moves no line between XCDs.
constexpr uint32_t kCtrStride = 128;

// A wave's view of a queue of n entries that all waves of the grid empty
// together. The queue is cut into chunks, the chunks into one contiguous
// segment per XCD (block b runs on XCD b % 8), and every wave starts with a
// chunk of its own, found without any atomic; the chunks beyond those are
// handed out by the segment's counter, and a wave whose segment is empty
// helps the others. A queue too short to give every lane of the grid an
// entry is spread over the waves: each works with fewer lanes, so that rays
// that would wait for one another in one wave run in several (4096 rays over
// 4096 waves 160 us, three to a wave 198 us).
// With the counters on one line, an atomic per 64 rays and eight more for
// every wave's end, the 1.6M closest-hit rays of a 256 x 256 x 8 Cornell
// generation took 2.27 ms; with this queue and trace_queue 0.62 ms.
//
// kStatic: no counters. The waves share the chunks out among themselves, wave
// w taking w, w + waves, ... , so calls that overlap on a stream share nothing.
template <bool kStatic>
struct WorkQueue {
  uint32_t n, chunk, chunks;
  uint32_t *ctr;
  uint32_t seg, base, limit;
  int lanes, refillMin;
  uint64_t laneMask;
  bool open;  // chunks may be left beyond the current one

  __device__ __forceinline__ uint32_t seg_lo(uint32_t x) const { return (uint32_t)(((uint64_t)chunks * x) / kXcds); }
  __device__ __forceinline__ uint32_t seg_waves(uint32_t x) const {
    return ((gridDim.x + (uint32_t)kXcds - 1u - x) / (uint32_t)kXcds) * (blockDim.x >> 6);
  }
  __device__ __forceinline__ bool set(uint32_t c) {
    base = c * chunk;
    limit = n - base < chunk ? n : base + chunk;
    return true;
  }

  // `reverse`: first chunks go to the waves from the grid's end, for the
  // second of two queues that one launch empties.
  __device__ __forceinline__ WorkQueue(uint32_t n_, uint32_t *ctr_, bool reverse) : n(n_), ctr(ctr_) {
    const uint32_t waves = gridDim.x * (blockDim.x >> 6);
    lanes = (int)queue_lanes(n, waves);
    chunk = queue_chunk(n, waves);
    chunks = queue_chunks(n, chunk);
    laneMask = lanes == 64 ? ~0ull : (1ull << lanes) - 1ull;
    refillMin = min(lanes, kRefill);
    seg = blockIdx.x % (uint32_t)kXcds;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rank = (blockIdx.x / (uint32_t)kXcds) * (blockDim.x >> 6) + wave;
    const uint32_t c = seg_lo(seg) + (reverse ? seg_waves(seg) - 1u - rank : rank);
    base = limit = 0;
    open = true;
    if (kStatic) {
      seg = blockIdx.x * (blockDim.x >> 6) + wave;
      if (seg < chunks) set(seg);
      return;
    }
    if (c < seg_lo(seg + 1u)) set(c);
  }

  // Entries left for this wave (fetches a chunk when the current one is used up).
  __device__ __forceinline__ bool more() {
    if (base < limit) return true;
    if (kStatic) {
      const uint32_t waves = gridDim.x * (blockDim.x >> 6);
      if (seg >= chunks || chunks - seg <= waves) return false;
      seg += waves;
      return set(seg);
    }
    while (open) {
      uint32_t first = seg_lo(seg) + seg_waves(seg), end = seg_lo(seg + 1u);
      if (first < end) {
        uint32_t c = 0;
        if (lane_id() == 0) c = atomicAdd(ctr + seg * kCtrStride, 1u);
        c = first + __builtin_amdgcn_readfirstlane(c);
        if (c < end) return set(c);
      }
      // This segment is empty: look for another that is not.
      const uint32_t x = (seg + lane_id()) % (uint32_t)kXcds;
      bool left = false;
      if (lane_id() < (uint32_t)kXcds) {
        const uint32_t f = seg_lo(x) + seg_waves(x), e = seg_lo(x + 1u);
        left = f < e && f + __hip_atomic_load(ctr + x * kCtrStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < e;
      }
      const uint64_t m = __ballot(left);
      open = m != 0ull;
      if (open) seg = (seg + (uint32_t)__builtin_ctzll(m)) % (uint32_t)kXcds;
    }
    return false;
  }
  // Hands out up to `want` entries from `first` on.
  __device__ __forceinline__ uint32_t take(uint32_t want, uint32_t &first) {
    const uint32_t k = min(want, limit - base);
    first = base;
    base += k;
    return k;
  }
};

}  // namespace mtx
