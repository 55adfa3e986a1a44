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

// x / T as the division rounds it, in three or four multiply-adds.
//
// With inv = 1 / T rounded to nearest and q within one unit in the last place
// of x / T, r = x - q T is exact and q + r inv rounds to x / T (Markstein's
// theorem; it excludes a T whose mantissa is all ones).  q = x inv is that
// close, 2^24 e + 1/2 units, for e = |inv T - 1| <= 2^-25 (`direct`, about three
// of four T).  Other T, e up to 2^-24, take lo = 1 / T - inv along: q = x inv +
// x lo, 1/2 unit and 2^-22.  x and every value between must stay in the normal
// range.
struct Quotient {
    float T, inv, lo;
    bool direct;
    __device__ __forceinline__ explicit Quotient(float t) : T(t), inv(1.0f / t) {
        const float e = __builtin_fmaf(-inv, t, 1.0f);  // exact
        lo = e * inv;
        direct = __builtin_fabsf(e) <= 0x1p-25f;
    }
    template <bool DIRECT>
    __device__ __forceinline__ float first(float x) const {
#pragma clang fp contract(off)
        return DIRECT ? x * inv : __builtin_fmaf(x, inv, x * lo);
    }
    template <bool DIRECT>
    __device__ __forceinline__ float of(float x) const {
        const float q = first<DIRECT>(x);
        return __builtin_fmaf(__builtin_fmaf(-q, T, x), inv, q);
    }
};

}  // namespace d3d
