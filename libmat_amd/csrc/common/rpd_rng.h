// The project's counter-based generator (host side): a draw is a hash of
// (seed, stream, index).
#pragma once

#include <stdint.h>

inline uint64_t rpd_mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

// One stream of a seed: the part of the hash that its draws share is
// computed once.
struct RpdRngStream {
  uint64_t key;
  RpdRngStream(uint64_t seed, uint64_t stream)
      : key(rpd_mix64(rpd_mix64(seed) ^ (stream * 0xD1B54A32D192ED03ULL))) {}
  uint64_t u64(uint64_t index) const { return rpd_mix64(key ^ index); }
  double uniform(uint64_t index) const {
    return (double)(u64(index) >> 11) * 0x1.0p-53;
  }
};
