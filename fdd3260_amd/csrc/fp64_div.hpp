// fp64_div.hpp -- FP64 divisions without the compiler's operand scaling, for
// the kernels that keep the reference's correctly rounded quotients.
#pragma once
#include <hip/hip_runtime.h>

namespace mimadv {

// FP64 division in the steps the compiler emits for n / d on gfx950
// (reciprocal estimate, two Newton steps, quotient, residual, corrected
// quotient) without its operand scaling and special-value fix-up.  Those
// two steps leave operands and result unchanged when n, d and n/d are
// normal numbers well inside the exponent range, so within that range the
// result is the correctly rounded quotient, bit for bit the same as n / d
// (checked on 3.4e10 random operand pairs in [2^-400, 2^400]).  A
// reciprocal serves every quotient with the same denominator.
__device__ __forceinline__ double refined_rcp(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    double e = fma(-d, r, 1.0);
    r = fma(r, e, r);
    e = fma(-d, r, 1.0);
    return fma(r, e, r);
}

__device__ __forceinline__ double quot(double n, double d, double r)
{
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}

// Residual classes that send a quotient to the plain division: NaN, infinite
// or subnormal.  With q = fl(n r) and an exact residual n - d q the corrected
// quotient is the rounded one; the residual is exact unless it falls below
// 2^-1022, where its class shows it (a residual that rounds to zero there
// means |n/d - q| is below half the spacing of q already).  n or q infinite
// or NaN gives a NaN residual.
constexpr int RES_BAD = 0x3 | 0x204 | 0x90;

// n / d with the refined reciprocal where the steps are exact, the plain
// division elsewhere (see refined_rcp, RES_BAD); exact zeros may lose their
// sign.
__device__ __forceinline__ double quotient(double n, double d)
{
    const double r = refined_rcp(d), q = n * r, e = fma(-d, q, n), a = fabs(d);
    double v = fma(e, r, q);
    if (__builtin_expect(!(a >= 0x1p-400 && a <= 0x1p400) || __builtin_amdgcn_class(e, RES_BAD), 0)) v = n / d;
    return v;
}

// Divisions by one positive denominator (a level thickness): one refined
// reciprocal, then three instructions and a class test per numerator.  A
// denominator outside the range of refined_rcp gets a NaN reciprocal, which
// the class test turns into plain divisions.  Exact zeros may lose their
// sign.
struct LevelDiv {
    double d, r;
    __device__ __forceinline__ explicit LevelDiv(double den)
        : d(den), r(den >= 0x1p-400 && den <= 0x1p400 ? refined_rcp(den) : __builtin_nan(""))
    {
    }
    // a denominator whose reciprocal was formed before
    __device__ __forceinline__ LevelDiv(double den, double rcp) : d(den), r(rcp) {}
    __device__ __forceinline__ double div(double n) const
    {
        const double q = n * r, e = fma(-d, q, n);
        double v = fma(e, r, q);
        if (__builtin_expect(__builtin_amdgcn_class(e, RES_BAD), 0)) v = n / d;
        return v;
    }
};

}  // namespace mimadv
