// When a double sum of floats does not depend on the order of its adds.
//
// Compiles as HIP device code and as plain C++ (the test build).
#pragma once

#include "bm_libm.h"

namespace bm {

// `sum`: non-negative floats added in double in any order; `least`: the
// smallest of them that is not zero.  Every term is a multiple of least's ulp
// u (2^-149 at least), and so is every sum of terms; multiples of u up to
// 2^53 u are doubles.  No partial sum exceeds the result (rounding is
// monotone), so with sum <= 2^53 u every add was exact, here and in any other
// order.
BM_HD bool exact_sum(double sum, float least) {
  const uint32_t e = libm::u32_of(least) >> 23;
  const uint64_t limit = (uint64_t)((e > 1 ? e : 1) - 127 - 23 + 53 + 1023) << 52;  // 2^53 u
  return sum <= libm::dbl_of(limit);
}

}  // namespace bm
