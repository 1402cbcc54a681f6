// Numbers by which a decode launch that folds its partials knows its own flags and words from whatever else the
// workspace holds.  Host code without HIP, so that the host tests can check the sequence.
#pragma once
#include <stdint.h>

namespace llmhip {

// The number after n.  All 2^64 come up once before one returns, and two launches also differ in either 32-bit half of their
// numbers unless 2.97e9 or more lie between them (2^64 over the golden ratio: its multiples keep the farthest apart).
// Numbers with a half of zero are left out: memory that was cleared holds neither half.
inline uint64_t next_launch_number(uint64_t n) {
  do n += 0x9E3779B97F4A7C15ull;
  while ((uint32_t)n == 0 || (uint32_t)(n >> 32) == 0);
  return n;
}

}  // namespace llmhip
