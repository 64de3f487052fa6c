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

// Entries of a chunk: one per lane, up to four in queues of thousands a wave.
constexpr uint32_t queue_chunk(uint32_t n, uint32_t waves) {
  const uint32_t lanes = queue_lanes(n, waves);
  if (lanes < 64u) return lanes;
  const uint64_t times = n / ((uint64_t)waves * 512u);
  return 64u * (times < 1u ? 1u : (times > 4u ? 4u : (uint32_t)times));
}

constexpr uint32_t queue_chunks(uint32_t n, uint32_t chunk) { return n / chunk + (n % chunk != 0u ? 1u : 0u); }

}  // namespace mtx
