// weno_ratio.hpp -- the smoothness-ratio switch of the reference 'weno'
// weights (advq_weno.f90:339-349: nonlinear weights when
// max(eta)/(min(eta)+eps) > 20) evaluated without the division but with the
// same outcome as the correctly rounded quotient.  Shared by the plain FP64
// forward kernel and the adjoint, so that both take the branch the CPU
// restatement takes.
#pragma once
#include <hip/hip_runtime.h>

namespace mimadv {

// fl(x/d) > T for T = 20 or 10 without the division, d > 0: the quotient
// rounds above T iff x/d > T + ulp(T)/2 (that tie rounds to the even T), i.e.
// iff x - T d > h = 2^-49 d (2^-50 d for T = 10).  Rounding is monotone and h
// is exact, so y = fl(x - T d) from one fma lies above (below) h only where
// the exact difference does; at y = h the division decides.
template <int T>
__device__ __forceinline__ bool ratio_above(double x, double d)
{
    static_assert(T == 20 || T == 10, "half an ulp of T");
    const double y = fma(-double(T), d, x);
    const double h = d * (T == 20 ? 0x1p-49 : 0x1p-50);
    bool r = y > h;
    if (__builtin_expect(y == h, 0)) r = x / d > double(T);
    return r;
}

__device__ __forceinline__ bool ratio_above_20(double x, double d) { return ratio_above<20>(x, d); }

}  // namespace mimadv
