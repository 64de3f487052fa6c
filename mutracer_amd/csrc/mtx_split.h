// How the waves of a grid share a queue of n entries: the counts that the
// kernels and the code that sizes their memory have to agree on. Holds for
// every 32-bit n.
#pragma once
#include <stdint.h>

namespace mtx {

// Lanes of a wave that take entries.
constexpr uint32_t queue_lanes(uint32_t n, uint32_t waves) {
  const uint64_t per = ((uint64_t)n + waves - 1u) / waves;
  return per < 1u ? 1u : (per > 64u ? 64u : (uint32_t)per);
}

// Entries of a chunk: one per lane, and up to four per lane where a wave takes
// more than 512 entries, so that a wave keeps to neighbouring rays. 1M-triangle
// 1080p step: 133.9 ms, with at most one per lane 136.7, sixteen 134.5, from
// 128 entries a wave on 134.7, from 2048 on 135.0. 16M camera rays in 24 x 60k
// triangles: 3.43, 3.95, 3.68, 3.42, 3.93 ms; 6M in 1M triangles 2.09, 2.21,
// 2.09, 2.21, 2.22; 4M scattered rays 9.18, 9.18, 9.18, 9.64, 9.18.
constexpr uint32_t queue_chunk(uint32_t n, uint32_t waves) {
  const uint32_t lanes = queue_lanes(n, waves);
  if (lanes < 64u) return lanes;
  const uint64_t times = n / ((uint64_t)waves * 512u);
  return 64u * (times < 1u ? 1u : (times > 4u ? 4u : (uint32_t)times));
}

constexpr uint32_t queue_chunks(uint32_t n, uint32_t chunk) { return n / chunk + (n % chunk != 0u ? 1u : 0u); }

}  // namespace mtx
