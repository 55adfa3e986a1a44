// Scalar arithmetic of the row passes, in plain C++ but for the exp2 that the
// caller hands in, so that a host compiler can sweep it.
#pragma once

namespace d3d {

// e^d for d in [-104, 0] (NaN for NaN), as 2^n 2^f: n = rint(d log2 e), f the
// rest, summed from the product's exact rounding error and the rest of log2 e,
// so that exp2's own error is all there is to speak of.  Without the range
// checks of expf, which the callers' d does not need.  exp2: 2^f for |f| <= 1/2,
// ldexp: p 2^n.
template <typename Exp2, typename Ldexp>
__device__ __forceinline__ float exp_reduced(float d, Exp2&& exp2, Ldexp&& ldexp) {
#pragma clang fp contract(off)
    constexpr float kLog2e = 1.44269502f, kLog2eRest = 1.92596299e-8f;
    const float t = d * kLog2e, n = __builtin_rintf(t);
    const float rest = __builtin_fmaf(d, kLog2eRest, __builtin_fmaf(d, kLog2e, -t));
    return ldexp(exp2((t - n) + rest), (int)n);
}

}  // namespace d3d
