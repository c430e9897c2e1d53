// Division by a number that is fixed for a launch, as a multiplication: plain integer code, the same on host and device.
#pragma once
#include <cstdint>

namespace sd {

// ceil(2^32 / d) if (v * that) >> 32 is v / d for every v below `below`, else 0.  With m = (2^32 + e) / d, e < d, the product is
// v / d + v * e / (d * 2^32): nothing is carried over to the next whole number while v * e < 2^32.
inline uint32_t exact_reciprocal(int64_t d, int64_t below) {
  if (d < 2 || d >= (1LL << 31) || below > (1LL << 32)) return 0;
  const int64_t m = ((1LL << 32) + d - 1) / d, e = m * d - (1LL << 32);
  return e == 0 || below <= (1LL << 32) / e ? (uint32_t)m : 0;
}

}  // namespace sd
