// Division by a run-time constant as a multiplication: the host prepares the
// reciprocal, the kernels get the quotient with one high product and a
// correction instead of the ~20 (32 bit) or ~100 (64 bit) instructions of a
// division.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hom {

// n / d for n < 2^32 given m = floor(2^32 / d) (0xffffffff for d == 1): the
// high product is the quotient or one less.
__device__ __forceinline__ uint32_t divByMagic(uint32_t n, uint32_t d,
                                               uint32_t m) {
  const uint32_t q = __umulhi(n, m);
  return n - q * d >= d ? q + 1 : q;
}
inline uint32_t magicFor(uint32_t d) {
  return d <= 1 ? 0xffffffffu : uint32_t((uint64_t(1) << 32) / d);
}

} // namespace hom
