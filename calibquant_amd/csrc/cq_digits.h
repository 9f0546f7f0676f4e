// Fixed-point operands of the 8-bit integer matrix instructions: numbers as four signed byte digits.  Plain C++, for host
// and device code alike.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define CQ_DIGITS __host__ __device__ __forceinline__
#else
#define CQ_DIGITS inline
#endif

namespace cq {

// four signed byte digits of x, -2^31 <= x <= 2^31 - 1 - 0x808080 (digit 0 in the lowest byte; above that the top digit wraps)
CQ_DIGITS uint32_t byte_digits(int x) { return (static_cast<uint32_t>(x) + 0x00808080u) ^ 0x00808080u; }

// A weight on its grid as digits: 0 <= e * grid <= 2^30, grid a power of two.  The product is exact and is rounded once, to the
// nearest whole number: off by half a step at most, and exact from 2^23 steps on.  (The conversion cuts off; the largest number below a half,
// added in the multiplication, makes that the nearest, and is too small to move a number of 2^23 steps.  Adding 0x808080 before
// the conversion as well would round what lies between 2^23 and 2^24 steps to an even number of them.)
CQ_DIGITS uint32_t weight_digits(float e, float grid) { return byte_digits(static_cast<int>(__builtin_fmaf(e, grid, 0.49999997f))); }

}  // namespace cq
