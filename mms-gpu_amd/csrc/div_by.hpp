// div_by.hpp -- the charge stencil's divisions by the cell sizes.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace mms {

// a / d for r = 1 / d rounded to nearest: the product a r corrected once by
// its remainder rounds like the division (Markstein's theorem) in four
// operations, the division's own sequence takes eleven.  div_fixup gives the
// division's results for zeros, infinities and NaN.  The remainder is exact
// while |a| > 2^-125; below, the last bit may differ.
__device__ __forceinline__ float div_by(float a, float d, float r) {
    const float q = a * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, a), r, q), d, a);
}

// cell sizes for which r and the products above stay normal numbers
inline bool div_by_ok(float d) { return d >= ldexpf(1.0f, -60) && d <= ldexpf(1.0f, 60); }

}  // namespace mms
