// Division by loop- or launch-invariant divisors as a multiply-high and a
// shift (Granlund & Montgomery, "Division by Invariant Integers using
// Multiplication", PLDI 1994, round-up variant), valid for 0 <= n, d < 2^31.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace spyre_hip {

struct FastDiv {
  uint32_t d, mul, shift;
};

inline FastDiv make_fastdiv(uint32_t d) {
  uint32_t l = 0;
  while ((uint64_t{1} << l) < d) ++l;
  const uint64_t m = ((uint64_t{1} << 32) * ((uint64_t{1} << l) - d)) / d + 1;
  return FastDiv{d, static_cast<uint32_t>(m), l};
}

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f) {
  return (__umulhi(n, f.mul) + n) >> f.shift;
}

}  // namespace spyre_hip
