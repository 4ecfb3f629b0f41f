// The exponential of the row softmax (gfx950).
#pragma once
#include <hip/hip_runtime.h>

namespace sddmm {

// exp(x) for x <= 0: 2^t with t = x log2(e) rounded, times 1 + (what the rounding of t and of log2(e) left out) ln 2.
// About one ulp; the library routine costs three times as much, and these passes would be bound by it.
__device__ __forceinline__ float exp_nonpositive(float x)
{
    x = x < -1000.f ? -1000.f : x;  // (0 from there on, for -infinity as well, which the next line would make a NaN)
    const float l2e = 1.44269502e+0f, l2e_lo = 1.92596299e-8f;
    const float t = x * l2e;
    const float r = fmaf(x, l2e_lo, fmaf(x, l2e, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, r * 0.693147182f, e);
}

}  // namespace sddmm
