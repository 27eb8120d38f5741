// div_by.hpp -- the charge stencil's divisions by the cell sizes.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace mms {

// a / d for r = 1 / d rounded to nearest: the product a r corrected once by
// its remainder rounds like the division (Markstein's theorem) in four
// operations, the division's own sequence takes eleven.  div_fixup gives the
// division's results for zeros, infinities, NaN and quotients beyond the
// float range.  The remainder's last bit is 2^-47 of a, so it is exact for
// |a| >= 2^-102 (and quotients that are normal numbers); below, the last bit
// may differ (on the CPU first at 2^-108 in 3.4e8 quotients of 414 divisors,
// 2% of them at 2^-123 for d = 5e-9).
__device__ __forceinline__ float div_by(float a, float d, float r) {
    const float q = a * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, a), r, q), d, a);
}

// cell sizes for which r and the products above stay normal numbers
inline bool div_by_ok(float d) { return d >= ldexpf(1.0f, -60) && d <= ldexpf(1.0f, 60); }

}  // namespace mms
