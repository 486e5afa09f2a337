// schemes_fp64.hpp -- per-face and per-cell device formulas of the MIMICA
// advection schemes, FP64, in the reference's floating-point operation order.
//
// The reference computes each direction as a sequential line sweep
// (face fluxes into a line array, then differences).  Here every formula
// is a pure function of a face or cell index and accessors Q(i), U(i)
// (1-based line indices), so a thread can evaluate one face (the marching
// kernels) or one cell (the PPM kernel) without the line sweep.  Position-dependent closures (tile
// edges, bottom/top levels) are selected by index exactly where the
// reference's loops switch formulas.  Built without FMA contraction these
// reproduce the reference arithmetic bit for bit.
#pragma once
#include <hip/hip_runtime.h>

#include "fp64_div.hpp"
#include "metric.hpp"
#include "weno_ratio.hpp"

namespace mimadv {

struct ZMetrics {
    const double *fdz0, *dzw, *dz1w, *dz1;
    const double *ppmc;  // [nz][12] PPM non-uniform coefficients per level
    const float *momz;   // [nz][MOMZ_N] level coefficients of the FP32 batched momentum operator
    double dz;
};

struct SchemeParams {
    int scheme;
    int muscl_limiter;
    int ppm_limiter;
    int weno_bottom;
    double lim_tol;
    double dt0;
};

__device__ __forceinline__ double dmaxd(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmind(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double sgn1(double x) { return copysign(1.0, x); }

// ---------------------------------------------------------------------------
// WENO5-JS (extension, no reference counterpart): Jiang & Shu (1996) left
// face value from a..e = x(f-2..f+2); eps = 1e-6, p = 2
// ---------------------------------------------------------------------------
__device__ __forceinline__ double weno5_left(double a, double b, double c, double d, double e)
{
    const double eps = 1e-6;
    double q0 = (2.0 * a - 7.0 * b + 11.0 * c) / 6.0;
    double q1 = (-b + 5.0 * c + 2.0 * d) / 6.0;
    double q2 = (2.0 * c + 5.0 * d - e) / 6.0;
    double b0 = 13.0 / 12.0 * (a - 2.0 * b + c) * (a - 2.0 * b + c) + 0.25 * (a - 4.0 * b + 3.0 * c) * (a - 4.0 * b + 3.0 * c);
    double b1 = 13.0 / 12.0 * (b - 2.0 * c + d) * (b - 2.0 * c + d) + 0.25 * (b - d) * (b - d);
    double b2 = 13.0 / 12.0 * (c - 2.0 * d + e) * (c - 2.0 * d + e) + 0.25 * (3.0 * c - 4.0 * d + e) * (3.0 * c - 4.0 * d + e);
    double a0 = 0.1 / ((eps + b0) * (eps + b0));
    double a1 = 0.6 / ((eps + b1) * (eps + b1));
    double a2 = 0.3 / ((eps + b2) * (eps + b2));
    return (a0 * q0 + a1 * q1 + a2 * q2) / (a0 + a1 + a2);
}

// ---------------------------------------------------------------------------
// MUSCL (advq_muscl.f90)
// ---------------------------------------------------------------------------

// limiter_muscl (advq_muscl.f90:335-383)
__device__ __forceinline__ void muscl_limiter(int lim, double lt, double xx, double ffip1, double ffip2,
                                              double ffim1, double &phir, double &phil)
{
    double rp1 = 1.0, rp2 = 1.0;
    if (fabs(ffim1) > lt * fabs(xx) && fabs(ffip1) < fabs(ffim1) / lt) rp1 = ffip1 / ffim1;
    if (fabs(ffip2) > lt * fabs(xx) && fabs(ffip1) < fabs(ffip2) / lt) rp2 = ffip1 / ffip2;
    switch (lim) {
    case 2:  // VL
        phil = (rp1 + fabs(rp1)) / (1.0 + fabs(rp1));
        phir = (rp2 + fabs(rp2)) / (1.0 + fabs(rp2));
        break;
    case 1:  // MC
        phil = dmaxd(0.0, dmind(dmind(2.0 * rp1, 0.5 * (rp1 + 1.0)), 2.0));
        phir = dmaxd(0.0, dmind(dmind(2.0 * rp2, 0.5 * (rp2 + 1.0)), 2.0));
        break;
    case 0:  // minmod
        phil = dmaxd(0.0, dmind(1.0, rp1));
        phir = dmaxd(0.0, dmind(1.0, rp2));
        break;
    default:  // Fromm
        phil = 0.5 * (rp1 + 1.0);
        phir = 0.5 * (rp2 + 1.0);
        break;
    }
}

__device__ __forceinline__ double muscl_upwind(double uu, double fl, double fr)
{
    return 0.5 * uu * (fl * (1.0 + sgn1(uu)) + fr * (1.0 - sgn1(uu)));
}

// |p| < |s| / lt (lt > 0) with the outcome of the rounded quotient: p lt and s
// differ by more than 2^-50 of s, or the division decides
__device__ __forceinline__ bool below_ratio(double p, double s, double lt)
{
    const double t = fma(-lt, fabs(p), fabs(s));
    bool r = t > 0.0;
    if (__builtin_expect(fabs(t) <= fabs(s) * 0x1p-50, 0)) r = fabs(p) < fabs(s) / lt;
    return r;
}

// Face flux from the two cell values, the slopes at the face and at its
// neighbours and the gate of the limiter.  `term(x)` scales a slope product to
// a value difference (x d in x and y, x / dz1w in z).
//
// The reference forms both sides' values and multiplies the off-side one by an
// exact zero, so with finite slopes the upwind side alone gives the flux (a
// zero may differ in sign); this halves the work and leaves one division of
// four (197 -> 168 us per launch at 256x256x128, 'MC').  Slopes that are not finite, or so large that a product may
// overflow, take the reference's sum, in which an infinite off side gives NaN.
template <class TF>
__device__ __forceinline__ double muscl_flux(const SchemeParams &sp, double uu, double xx, double xp, double slope_p,
                                             double slope_p2, double slope_m, bool limited, TF term)
{
    const double lt = sp.lim_tol;
    if (__builtin_expect(!(fabs(slope_m) + fabs(slope_p2) < 0x1p400 && fabs(slope_p) < 0x1p400), 0)) {
        double phir, phil, fl, fr;
        if (limited) {
            muscl_limiter(sp.muscl_limiter, lt, xx, slope_p, slope_p2, slope_m, phir, phil);
            fr = xp - term(0.5 * phir * slope_p2);
            fl = xx + term(0.5 * phil * slope_m);
        } else {
            fr = xp - term(0.5 * slope_p);
            fl = xx + term(0.5 * slope_p);
        }
        return muscl_upwind(uu, fl, fr);
    }
    const bool pos = !signbit(uu);
    const double so = pos ? slope_m : slope_p2, base = pos ? xx : xp;
    double v = 0.5 * slope_p;
    if (limited) {
        double r = 1.0;
        if (fabs(so) > lt * fabs(xx) && below_ratio(slope_p, so, lt)) r = quotient(slope_p, so);
        double phi;
        switch (sp.muscl_limiter) {
        case 2: phi = (r + fabs(r)) / (1.0 + fabs(r)); break;                                 // VL
        case 1: phi = fmax(0.0, fmin(fmin(2.0 * r, 0.5 * (r + 1.0)), 2.0)); break;            // MC
        case 0: phi = fmax(0.0, fmin(1.0, r)); break;                                         // minmod
        default: phi = 0.5 * (r + 1.0); break;                                                // Fromm
        }
        v = 0.5 * phi * so;
    }
    v = term(v);
    return uu * (pos ? base + v : base - v);
}

// face flux i+1/2, x/y (advq_muscl.f90:81-100)
template <class QF, class UF>
__device__ __forceinline__ double muscl_hface(int i, double d, double d1, const SchemeParams &sp, QF Q, UF U)
{
    const double eps = 1.e-18;
    double uu = U(i + 1), xx = Q(i);
    double xp = Q(i + 1);
    double slope_p = (xp - xx) * d1;
    double slope_p2 = (Q(i + 2) - xp) * d1;
    double slope_m = (xx - Q(i - 1)) * d1;
    const double gate = sp.lim_tol * fabs(xx) + eps;
    const bool limited = (d * fabs(slope_m) > gate) | (d * fabs(slope_p2) > gate);
    return muscl_flux(sp, uu, xx, xp, slope_p, slope_p2, slope_m, limited, [&](double x) { return x * d; });
}

// z face flux k+1/2 (advsz_muscl, advq_muscl.f90:245-302)
template <class QF, class WF>
__device__ __forceinline__ double muscl_zface(int f, int nz, const ZMetrics &zm, const SchemeParams &sp,
                                              double bc51, double bc61, QF Q, WF W)
{
    const double eps = 1.e-18;
    double dz = zm.dz;
    const auto dz1 = table(zm.dz1), fdz0 = table(zm.fdz0);
    const LevelDiv m(table(zm.dz1w)[f - 1]);
    const double xx = Q(f), xp = Q(f + 1), gate = sp.lim_tol * fabs(xx) + eps;
    const double slope_p = (xp - xx) * dz1[f - 1];
    double slope_p2, slope_m;
    bool limited;
    if (f == 1) {
        slope_p2 = (Q(3) - xp) * dz1[1];
        slope_m = bc51 * (Q(nz - 4) - Q(nz - 5)) * dz1[nz - 6] + (1.0 - bc51) * slope_p;
        limited = fdz0[1] * dz * fabs(slope_p2) > gate;
    } else if (f == nz - 1) {
        slope_m = (xx - Q(f - 1)) * dz1[f - 2];
        slope_p2 = bc61 * (Q(6) - Q(5)) * dz1[4] + (1.0 - bc61) * slope_p;
        limited = fdz0[f - 2] * dz * fabs(slope_m) > gate;
    } else {
        slope_m = (xx - Q(f - 1)) * dz1[f - 2];
        slope_p2 = (Q(f + 2) - xp) * dz1[f];
        limited = (fdz0[f - 2] * dz * fabs(slope_m) > gate) | (fdz0[f] * dz * fabs(slope_p2) > gate);
    }
    return muscl_flux(sp, W(f + 1), xx, xp, slope_p, slope_p2, slope_m, limited,
                      [&](double x) { return m.div(x); });
}

// ---------------------------------------------------------------------------
// QUICK (advq_quick.f90) and its unlimited form (advq_quick_nolim.f90)
// ---------------------------------------------------------------------------

// limiter_quick (advq_quick.f90:313-352); phic: x in x/y, x/dz in z
__device__ __forceinline__ void quick_limiter(double lt, double phic, double ffip1, double ffip2, double ffim1,
                                              double &phil, double &phir)
{
    const double eps = 1.e-18, c1 = 1.0 / 3.0;
    double rp1 = 1.0, rp2 = 1.0, rp11 = 1.0, rp21 = 1.0;
    if (fabs(ffim1) > lt * fabs(phic) + eps) rp1 = ffip1 / ffim1;
    if (fabs(ffip2) > lt * fabs(phic) + eps) rp2 = ffip1 / ffip2;
    if (fabs(ffip1) > lt * fabs(phic) + eps) {
        rp11 = ffim1 / ffip1;
        rp21 = ffip2 / ffip1;
    }
    phil = rp1 * (1.0 - c1 * (1.0 - rp11));
    phir = rp2 * (1.0 - c1 * (1.0 - rp21));
    if (fabs(ffim1) > lt * fabs(phic) + eps || fabs(ffip2) > lt * fabs(phic) + eps) {
        phil = dmaxd(0.0, dmind(2.0 * rp1, dmind(phil, 2.0)));
        phir = dmaxd(0.0, dmind(2.0 * rp2, dmind(phir, 2.0)));
    }
}

__device__ __forceinline__ double half_upwind(double uu, double fl, double fr)
{
    return 0.5 * fl * (uu + fabs(uu)) + 0.5 * fr * (uu - fabs(uu));
}

// face flux i+1/2, x/y (advq_quick.f90:75-88, advq_quick_nolim.f90:77-90)
template <bool NL, class QF, class UF>
__device__ __forceinline__ double quick_hface(int i, const SchemeParams &sp, QF Q, UF U)
{
    double uu = U(i + 1), xx = Q(i), xp = Q(i + 1);
    double ffip1 = xp - xx;
    double ffip2 = Q(i + 2) - xp;
    double ffim1 = xx - Q(i - 1);
    double phil, phir, fl, fr;
    if constexpr (NL) {
        const double cc = 1.0 / 4.0;
        phil = ffip1 - cc * (ffip1 - ffim1);
        phir = ffip1 + cc * (ffip2 - ffip1);
        fl = xx + 0.5 * phil;
        fr = xp - 0.5 * phir;
    } else {
        quick_limiter(sp.lim_tol, xx, ffip1, ffip2, ffim1, phil, phir);
        fl = xx + 0.5 * phil * ffim1;
        fr = xp - 0.5 * phir * ffip2;
    }
    return half_upwind(uu, fl, fr);
}

// bottom/core/top slopes of a z face (per metre), with the periodic-floor
// and periodic-lid substitutions of advsz_quick/advsz_lw
template <class QF>
__device__ __forceinline__ void z_slopes(int f, int nz, const ZMetrics &zm, double bc51, double bc61, QF Q,
                                         double ffip1, double &ffip2, double &ffim1)
{
    const auto dz1 = table(zm.dz1);
    if (f == 1) {
        ffip2 = (Q(3) - Q(2)) * dz1[1];
        ffim1 = bc51 * (Q(nz - 4) - Q(nz - 5)) * dz1[nz - 6] + (1.0 - bc51) * ffip1;
    } else if (f == nz - 1) {
        ffim1 = (Q(f) - Q(f - 1)) * dz1[f - 2];
        ffip2 = bc61 * (Q(6) - Q(5)) * dz1[4] + (1.0 - bc61) * ffip1;
    } else {
        ffip2 = (Q(f + 2) - Q(f + 1)) * dz1[f];
        ffim1 = (Q(f) - Q(f - 1)) * dz1[f - 2];
    }
}

// z face flux k+1/2 (advq_quick.f90:233-284, advq_quick_nolim.f90:239-286)
template <bool NL, class QF, class WF>
__device__ __forceinline__ double quick_zface(int f, int nz, const ZMetrics &zm, const SchemeParams &sp,
                                              double bc51, double bc61, QF Q, WF W)
{
    double xx = Q(f), ww = W(f + 1), xp = Q(f + 1);
    double ffip1 = (xp - xx) * table(zm.dz1)[f - 1];
    double ffip2, ffim1;
    z_slopes(f, nz, zm, bc51, bc61, Q, ffip1, ffip2, ffim1);
    const double m = table(zm.dz1w)[f - 1];
    double phil, phir, fl, fr;
    if constexpr (NL) {
        const double cc = 1.0 / 4.0;
        phil = ffip1 - cc * (ffip1 - ffim1);
        phir = ffip1 + cc * (ffip2 - ffip1);
        fl = xx + 0.5 * phil / m;
        fr = xp - 0.5 * phir / m;
    } else {
        quick_limiter(sp.lim_tol, xx / zm.dz, ffip1, ffip2, ffim1, phil, phir);
        fl = xx + 0.5 * phil * ffim1 / m;
        fr = xp - 0.5 * phir * ffip2 / m;
    }
    return half_upwind(ww, fl, fr);
}

// ---------------------------------------------------------------------------
// Lax-Wendroff (advq_lw.f90, limiter 'MC': the module's lwlimiter, which
// nothing in the model changes) and its unlimited form (advq_lw_nolim.f90)
// ---------------------------------------------------------------------------

// limiter_lw, 'MC' (advq_lw.f90:349-373,389-391)
__device__ __forceinline__ void lw_limiter(double lt, double xx, double ffip1, double ffip2, double ffim1,
                                           double &phir, double &phil)
{
    const double eps = 1.e-18;
    double rp1 = 1.0, rp2 = 1.0;
    if (fabs(ffim1) > lt * fabs(xx) + eps) rp1 = ffip1 / ffim1;
    if (fabs(ffip2) > lt * fabs(xx) + eps) rp2 = ffip1 / ffip2;
    phil = dmaxd(dmind(dmind(2.0 * rp1, 0.5 * (rp1 + 1.0)), 2.0), 0.0);
    phir = dmaxd(dmind(dmind(2.0 * rp2, 0.5 * (rp2 + 1.0)), 2.0), 0.0);
}

__device__ __forceinline__ double lw_flux(double uu, double fl, double fr)
{
    return 0.5 * uu * (fl * (sgn1(uu) + 1.0) - fr * (sgn1(uu) - 1.0));
}

// face flux i+1/2, x/y (advq_lw.f90:81-98, advq_lw_nolim.f90:79-88);
// Courant number from the full step dt0
template <bool NL, class QF, class UF>
__device__ __forceinline__ double lw_hface(int i, double d1, const SchemeParams &sp, QF Q, UF U)
{
    const double eps = 1.e-18;
    double uu = U(i + 1), xx = Q(i), xp = Q(i + 1);
    double ffip1 = xp - xx;
    double mu = fabs(uu) * sp.dt0 * d1;
    double fl, fr;
    if constexpr (NL) {
        fl = xx + 0.5 * ffip1 * (1.0 - mu);
        fr = xp - 0.5 * ffip1 * (1.0 - mu);
        return half_upwind(uu, fl, fr);
    }
    double ffim1 = xx - Q(i - 1);
    double ffip2 = Q(i + 2) - xp;
    double lt = sp.lim_tol;
    if (fabs(ffim1) > lt * fabs(xx) + eps || fabs(ffip2) > lt * fabs(xx) + eps) {
        double phir, phil;
        lw_limiter(lt, xx, ffip1, ffip2, ffim1, phir, phil);
        fl = xx + 0.5 * phil * ffim1 * (1.0 - mu);
        fr = xp - 0.5 * phir * ffip2 * (1.0 - mu);
    } else {
        fl = xx + 0.5 * ffip1 * (1.0 - mu);
        fr = xp - 0.5 * ffip1 * (1.0 - mu);
    }
    return lw_flux(uu, fl, fr);
}

// z face flux k+1/2 (advq_lw.f90:245-316, advq_lw_nolim.f90:226-235)
template <bool NL, class QF, class WF>
__device__ __forceinline__ double lw_zface(int f, int nz, const ZMetrics &zm, const SchemeParams &sp, double bc51,
                                           double bc61, QF Q, WF W)
{
    const double eps = 1.e-18;
    double xx = Q(f), ww = W(f + 1), xp = Q(f + 1);
    double mu = fabs(ww) * sp.dt0 * table(zm.dz1)[f - 1];
    double ffip1 = (xp - xx) * table(zm.dz1)[f - 1];
    const double m = table(zm.dz1w)[f - 1];
    double fl, fr;
    if constexpr (NL) {
        fl = xx + 0.5 * ffip1 * (1.0 - mu) / m;
        fr = xp - 0.5 * ffip1 * (1.0 - mu) / m;
        return half_upwind(ww, fl, fr);
    }
    double ffip2, ffim1;
    z_slopes(f, nz, zm, bc51, bc61, Q, ffip1, ffip2, ffim1);
    double lt = sp.lim_tol, dz = zm.dz;
    if (dz * fabs(ffim1) > lt * fabs(xx) + eps || dz * fabs(ffip2) > lt * fabs(xx) + eps) {
        double phir, phil;
        lw_limiter(lt, xx, ffip1, ffip2, ffim1, phir, phil);
        fl = xx + 0.5 * phil * ffim1 * (1.0 - mu) / m;
        fr = xp - 0.5 * phir * ffip2 * (1.0 - mu) / m;
    } else {
        fl = xx + 0.5 * ffip1 * (1.0 - mu) / m;
        fr = xp - 0.5 * ffip1 * (1.0 - mu) / m;
    }
    return lw_flux(ww, fl, fr);
}

// ---------------------------------------------------------------------------
// PPM (advq_ppm.f90)
// ---------------------------------------------------------------------------

// |x| > sqrt(spacing(x)) of Fortran for REAL(8), spacing = 2**(ilogb(x)-52)
// (2**-1022 at least): the root is 2**((e-52)/2) for an even exponent e of x
// and fl(sqrt(2)) 2**((e-53)/2) for an odd one, so it lies above |x| for e <=
// -54, at fl(sqrt(2)) 2**-53 for e = -53, at 2**-52 for e = -52 and below |x|
// from e = -51 on (false for infinities and NaN, whose root is infinite or
// undefined).
__device__ __forceinline__ bool above_sqrt_spacing(double x)
{
    const double a = fabs(x);
    return a > 0x1.6a09e667f3bcdp-53 && a != 0x1p-52 && a < __builtin_inf();
}

struct PPMRec {
    double fr, fl;
};

// smoothness of two neighbouring differences (advq_ppm.f90:449-530)
__device__ __forceinline__ double ppm_gamma(double a, double b)
{
    const double d = a - b, s = a + b;
    return 0.5 * (d * d + s * s);
}

// limiter_ppm (advq_ppm.f90:449-530) followed by the CW84 face averages
// Flux_r/Flux_l (advq_ppm.f90:93-94) of a cell: its value and neighbours, the
// right and left face values, the four differences around it, gamma1..3 =
// ppm_gamma of (ffip1, ffim1), (ffip2, ffip1), (ffim1, ffim2).  The
// conditions are formed without short-circuits (a branch per term costs more
// than the terms).
__device__ __forceinline__ PPMRec ppm_cell(int use_lim, double xx, double xp, double xm, double xplus, double xmin,
                                           double ffip1, double ffip2, double ffim1, double ffim2, double gamma1,
                                           double gamma2, double gamma3, double mup, double muc)
{
    const double eps = 1.e-15;
    double phir = xplus, phil = xmin;
    // a NaN among the gammas comes with a NaN face value, which stays
    const double gmax = fmax(fmax(gamma1, gamma2), gamma3), gmin = fmin(fmin(gamma1, gamma2), gamma3) + eps;
    double phi1 = phir - phil;
    double phi2 = 3.0 * (phil - 2.0 * xx + phir);
    // lambda = gmax / gmin > 10 without the division
    if (use_lim && ratio_above<10>(gmax, gmin)) {
        const bool turn = ffip1 * ffim1 <= 0.0;
        const bool wr = (phir < 0.0) | (((phir - xx) * (xp - phir) < 0.0) &
                                        ((ffim1 * ffip2 >= 0.0) | turn | (ffip2 * ffip1 <= 0.0)));
        const double nr = (fabs(phir - xx) < fabs(phir - xp)) ? xx : xp;
        const bool wl = (phil < 0.0) | (((xx - phil) * (phil - xm) < 0.0) &
                                        ((ffim2 * ffip1 >= 0.0) | (ffim2 * ffim1 <= 0.0) | turn));
        const double nl = (fabs(phil - xx) < fabs(phil - xm)) ? xx : xm;
        phir = wr ? nr : phir;
        phil = wl ? nl : phil;
        phi1 = phir - phil;
        phi2 = 3.0 * (phil - 2.0 * xx + phir);
        // slope = -phi1 / (2 sgn(phi2) max(|phi2|, eps)); the reference's
        // (slope > -1/2 .or. slope < 1/2) holds for every slope but NaN,
        // which takes phi1 NaN or an infinite phi1 over an infinite phi2
        const double inf = __builtin_inf();
        const bool slope_ok = (fabs(phi1) < inf) | ((phi1 == phi1) & (fabs(phi2) < inf));
        if ((fabs(phi2) > eps) & slope_ok) {
            // the ratio is finite or infinite here, not NaN
            const double rp1 = above_sqrt_spacing(ffim1) ? quotient(ffip1, ffim1) : 1.0;
            const double lim = fmax(0.0, fmin(fmin(2.0, 0.5 * (rp1 + 1.0)), 2.0 * rp1));
            const double r = xx + 0.5 * ffim1 * lim, l = xx - 0.5 * ffim1 * lim;
            const bool flat = (xx - l) * (r - xx) < 0.0;
            phir = flat ? xx : r;
            phil = flat ? xx : l;
            phi1 = phir - phil;
            phi2 = 0.0;
        }
    }
    PPMRec r;
    r.fr = phir - 0.5 * mup * (phi1 + (1.0 - (2.0 / 3.0) * mup) * phi2);
    r.fl = phil + 0.5 * muc * (phi1 - (1.0 - (2.0 / 3.0) * muc) * phi2);
    return r;
}

// Flux_r/Flux_l of cell c in 3..n-1 on an x/y line (advq_ppm.f90:79-134) from
// its five values and the Courant numbers; EDGE: the tile touches a side, so
// c may be 3 or n-1, whose closures take the nearer differences
template <bool EDGE>
__device__ __forceinline__ PPMRec ppm_hcell(int c, int n, const SchemeParams &sp, double qm2, double xm, double xx,
                                            double xp, double qp2, double mup, double muc)
{
    const bool lo = EDGE && c == 3, hi = EDGE && c == n - 1;
    const double ffip1 = xp - xx, ffim1 = xx - xm;
    const double ffip2 = hi ? ffip1 : qp2 - xp, ffim2 = lo ? ffim1 : xm - qm2;
    const double sl = 0.5 * (ffip1 + ffim1);  // also the slope of c-1 at its right
    const double xr = xx + 0.5 * ffip1, xl = xm + 0.5 * ffim1;
    double xplus = xr - (1.0 / 6.0) * (0.5 * (ffip2 + ffip1) - sl);
    double xmin = xl - (1.0 / 6.0) * (sl - 0.5 * (ffim1 + ffim2));
    if (lo | hi) xplus = xr;
    if (EDGE && c == 4) xmin = xl;
    if (lo) xmin = 0.5 * (xp + xx);
    return ppm_cell(sp.ppm_limiter, xx, xp, xm, xplus, xmin, ffip1, ffip2, ffim1, ffim2, ppm_gamma(ffip1, ffim1),
                    ppm_gamma(ffip2, ffip1), ppm_gamma(ffim1, ffim2), mup, muc);
}

__device__ __forceinline__ double ppm_faceflux(double fr, double fl, double uf)
{
    return 0.5 * fr * (uf + fabs(uf)) + 0.5 * fl * (uf - fabs(uf));
}

// Right-face value of level c (advq_ppm.f90:368-409) from its value x and the
// differences D(c-1), D(c), D(c+1), D(m) = Q(m+1) - Q(m).  Per-level
// coefficients (metric-only subexpressions of the non-uniform face formula,
// advq_ppm.f90:379-383, evaluated in the same order):
//  [0] delta/(dm1+delta+dp1)   [1] (2dm1+delta)/(dp1+delta)  [2] (delta+2dp1)/(dm1+delta)
//  [3] dp1/(delta+dp1+dp2)     [4] (2delta+dp1)/(dp2+dp1)    [5] (dp1+2dp2)/(delta+dp1)
//  [6] delta/(delta+dp1)       [7] 1/(dm1+delta+dp1+dp2)
//  [8] 2dp1*delta/(delta+dp1)*((dm1+delta)/(2delta+dp1)-(dp2+dp1)/(2dp1+delta))
//  [9] delta*(dm1+delta)/(2delta+dp1)   [10] dp1*(dp1+dp2)/(2dp1+delta)
__device__ __forceinline__ double ppm_zxplus(int c, int nz, Table<double> ppmc, double x, double dm, double d, double dp)
{
    if (c <= 2 || c == nz - 1) return x + 0.5 * d;
    const auto p = ppmc + 12 * (c - 1);
    const double sl = p[0] * (p[1] * d + p[2] * dm);
    const double slp1 = p[3] * (p[4] * dp + p[5] * d);
    return x + p[6] * d + p[7] * (p[8] * d - p[9] * slp1 + p[10] * sl);
}

}  // namespace mimadv
