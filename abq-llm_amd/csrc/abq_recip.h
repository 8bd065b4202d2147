// The correctly rounded reciprocal of a normal fp32 number from an estimate of it.  Plain C++, compiled for the device and,
// by the unit tests, for the host.
#pragma once
#include "abq_bits.h"

namespace abq {

// Two Newton steps in fp64 from an estimate whose relative error is at most 2^-20: the first leaves 2^-40, the second 2^-52
// (its own rounding).  A product of s and the midpoint m of two neighbouring floats, 24 and 25 significant bits, is never a
// power of two (m is odd), so 1 / s lies at least 2^-49 of its value away from every such m, and the conversion rounds as the
// exact quotient would.  Nothing depends on how good the hardware's estimate is beyond its stated 1 ulp (2^-22), and the chain
// is four fma in front of a row's codes where a full fp64 division is some forty instructions.  (One step in fp32 is not
// enough: from an estimate one ulp off it misses the rounded value for several mantissas, 0x7fffff among them.)
ABQ_HD float rounded_reciprocal(float s, float estimate)
{
    const double d = s;
    double r = estimate;
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    return (float)r;
}

} // namespace abq
