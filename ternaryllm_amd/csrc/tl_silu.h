// The SiLU of a product's gate, alike in every kernel that applies it.
#pragma once
#include <hip/hip_runtime.h>

namespace tl {

// g / (1 + exp(-g)), in every bit what the division gives (compared for all 2^32 values of g): an approximate quotient corrected by its
// own remainder, which a fused multiply-add has exactly (Markstein's step).  Bound by what is issued: eight instructions where hipcc's
// division takes some ten.  8192 x 2048 -> 11008 gated, in one run, 254 us / 250, and 247 with the quotient as it is, which is a unit off
// in one of 40.
// (A quarter of the denominator is inverted: the unit's results below 2^-126 are zero.)
__device__ __forceinline__ float silu(float g)
{
    const float d = 1.0f + __expf(-g), r = 0.25f * __builtin_amdgcn_rcpf(0.25f * d), q = g * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, g), r, q), d, g);   // (infinite g and d, and the sign of zero)
}

}  // namespace tl
