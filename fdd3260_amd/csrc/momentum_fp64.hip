// momentum_fp64.hip -- momentum flux divergence (qnadv_uvw) on gfx950.
//
// Restates src/INTEG/windadv.f90: flux-form centred differences of the
// momenta (rho0 u, rho0 v, rho0 w) advected by wind_adv, 2nd or 4th order
// (mom_ord), with the 4th-difference artificial viscosity (lavisc, avisc =
// 1/16) and the nnf/ope vertical closures.  The reference sweeps lines per
// direction and accumulates into ua in the order x,y,z (even ntime) or
// z,y,x (odd ntime, windadv.f90:103,158); here every cell adds the same
// per-direction increments in the same order.  Output arrays are overwritten
// everywhere (ghosts and w(k=1) get 0, as `ua = 0.0` at windadv.f90:97).
//
// Compiled with -ffp-contract=off to keep the reference operation order: the
// results are the reference arithmetic's bit for bit.
#include <type_traits>

#include "fp64_div.hpp"
#include "mimadv_internal.hpp"

namespace mimadv {

namespace {

constexpr double AVISC = 1.0 / 16.0;
constexpr int MOM_GROUPS = 3;  // resident work items per CU

struct MomCoefs {
    double c1s, c2s;           // self lines (4/3, 1/3)
    double c1c, c2c;           // cross lines (9/8, 1/8)
    double dx1, dx2, dx3;      // 1/dx, 1/(2 dx), 1/(3 dx)
    double dy1, dy2, dy3;
};

__device__ __forceinline__ double visc5(const double *m)  // m[0..4] = M(i-2..i+2)
{
    return -m[4] + 4.0 * m[3] - 6.0 * m[2] + 4.0 * m[1] - m[0];
}

// advux_fd / advvy_fd: self advection along a line (windadv.f90:526-548)
// added to t; m, u[0..4] = values at i-2..i+2
template <bool VISC>
__device__ __forceinline__ double self_line(double t, const double *m, const double *u, double d1, double d2,
                                            const MomCoefs &c)
{
    auto flux = [&](int n) { return ((u[n + 1] + u[n]) * 0.5) * ((m[n + 1] + m[n]) * 0.5); };
    auto advf = [&](int n) { return ((u[n + 2] + u[n]) * 0.5) * ((m[n + 2] + m[n]) * 0.5); };
    t = t + c.c1s * (flux(2) - flux(1)) * d1 - c.c2s * (advf(2) - advf(0)) * d2;
    if constexpr (VISC) t = t - AVISC * (fabs(u[2]) * d1) * visc5(m);
    return t;
}

// four-point average of the advecting component across the line (or, for the
// vertical momentum, across levels): near pair n1 + n2, far pair f1 + f2
__device__ __forceinline__ double interp4(const MomCoefs &c, double n1, double n2, double f1, double f2)
{
    return c.c1c * (n1 + n2) * 0.5 - c.c2c * (f1 + f2) * 0.5;
}

// advuy_fd / advvx_fd (windadv.f90:587-620) and advwx_fd / advwy_fd
// (:927-962) added to t: m[0..4] = M(i-2..i+2), vv[0..3] = the averaged
// advecting component at i-1..i+2, mus the four velocities of the viscosity,
// summed
template <bool VISC>
__device__ __forceinline__ double cross_line(double t, const double *m, const double *vv, double mus, double d1,
                                             double d3, const MomCoefs &c)
{
    auto flux = [&](int n) { return vv[n] * ((m[n + 1] + m[n]) * 0.5); };  // face i-2+n + 1/2
    t = t + c.c1c * (flux(2) - flux(1)) * d1 - c.c2c * (flux(3) - flux(0)) * d3;
    if constexpr (VISC) t = t - AVISC * (0.25 * fabs(mus) * d1) * visc5(m);
    return t;
}

// The vertical terms of a component added to t.  With flux(0) and flux(nz) set
// by the boundary (see momentum_march_kernel) every closure of
// windadv.f90:656-688 and :1077-1121 is a selection by level: the first and
// last level take the plain difference (coefficient 1, no wide term), 'per'
// floors and lids add nothing, the viscosity acts on levels 3..nz-2.
struct LevelZ {
    bool mid, on, visc;
    __device__ __forceinline__ LevelZ(int k, int nz, int bc5, int bc6)
        : mid(k >= 2 && k < nz), on(k <= 2 ? bc5 != 0 : (k == nz ? bc6 != 0 : true)), visc(k >= 3 && k <= nz - 2)
    {
    }
    // near, far: flux differences; c1, c2 their coefficients; m the metric of
    // the near term, d the thickness of the wide one; mu the viscosity speed
    template <bool VISC>
    __device__ __forceinline__ double add(double t, double near, double far, double c1, double c2, double m,
                                          const LevelDiv &d, double mu, const double *mz) const
    {
        if (on) {
            if (mid) t = t + c1 * near * m - d.div(c2 * far);
            else t = t + near * m;
        }
        if constexpr (VISC) {
            if (visc) t = t - AVISC * mu * visc5(mz);
        }
        return t;
    }
};

// Levels of a work item at most (the metrics of its levels sit in LDS).
constexpr int MOM_LEVELS = 16;

// One work item: a TX x TY column tile marched up a chunk of levels.
//
// What bounds it: FP64 issue (about 520 vector instructions per cell, 72 LDS
// reads) at three waves per SIMD, not its 72 bytes per cell, so every value is
// formed once.  Per level the six arrays go through LDS with a 2-cell halo;
// the advecting components averaged across the lines (lvx, luy) or across
// levels (luu, lvv) are formed once per point instead of once per face that
// uses them (four); the vertical fluxes are carried up the column in registers
// instead of being formed four times; the metric divisions share one
// reciprocal per level, kept in LDS.  51.6 KB of LDS and 168 VGPRs: three
// groups per CU without spills (the components are fenced from each other by
// settle(), otherwise 350 VGPRs are wanted).
//
// Measured, mom_ord 4 with viscosity, against one thread per cell that
// recomputes every flux from global memory with full divisions: 256x256x128
// 2300 -> 280 us (2.2 TB/s of its 72 B per cell), 64x64x48 86 -> 22 us.
template <int TX, int TY, bool VISC, bool EVEN>
__global__ __launch_bounds__(TX *TY) __attribute__((amdgpu_waves_per_eu(3, 8))) void momentum_march_kernel(
    GridDev g, MomCoefs c, const double *__restrict__ mu, const double *__restrict__ mv, const double *__restrict__ mw,
    const double *__restrict__ ut, const double *__restrict__ vt, const double *__restrict__ wt,
    const double *__restrict__ dzw, const double *__restrict__ dz1w, const double *__restrict__ dz1,
    double *__restrict__ ua, double *__restrict__ va, double *__restrict__ wa, int kchunk, int ntx, int nwork)
{
    constexpr bool THREE_D = TY > 1;
    constexpr int NT = TX * TY, H = 2;
    constexpr int LW = TX + 2 * H, LH = THREE_D ? TY + 2 * H : 1, PL = LW * LH;
    constexpr int TS = (PL + NT - 1) / NT;
    constexpr int NVX = THREE_D ? TX * (TY + 3) : 1;  // vvx rows j0-1..j0+TY+1
    constexpr int UW = TX + 3, NUY = THREE_D ? UW * TY : 1;  // uuy columns i0-1..i0+TX+1
    __shared__ double lmu[PL], lmv[THREE_D ? PL : 1], lmw[PL];  // level k
    __shared__ double rut[4][PL], rvt[THREE_D ? 4 : 1][PL];     // rings of the levels k-2..k+1
    __shared__ double lw[PL];                                   // wt at level k+2
    __shared__ double luu[UW * TY], lvv[NVX];  // ut, vt averaged to the w level k, at the columns w reads
    __shared__ double luy[NUY], lvx[NVX];      // ut averaged in y, vt averaged in x, level k
    // metrics of the levels k0-1..k1+1: thickness, thickness of the pair
    // (k, k+1) and its reciprocal, of (k-1, k, k+1) and its reciprocal,
    // dz1w(k), dz1(k-1), thickness of k+1
    constexpr int NM = 8;
    __shared__ double lmet[(MOM_LEVELS + 2) * NM];

    const int nx = g.nx, ny = g.ny, nz = g.nz, bc5 = g.bcl[4], bc6 = g.bcl[5];
    const size_t plane = (size_t)nx * ny;
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int nchunk = (nz + kchunk - 1) / kchunk, ntile = nwork / nchunk;
    // chunks outermost, tiles x-fastest; the hardware deals groups round-robin
    // over the 8 XCDs, so each XCD gets a contiguous range of the list and
    // neighbouring tiles share their halo rows in one L2
    const int wi = blockIdx.x;
    const int wk = (nwork % 8 == 0) ? (wi % 8) * (nwork / 8) + wi / 8 : wi;
    const int kc = wk / ntile, tile = wk - kc * ntile;
    const int i0 = 4 + (tile % ntx) * TX, j0 = THREE_D ? 4 + (tile / ntx) * TY : 1;
    const int k0 = 1 + kc * kchunk, k1 = min(nz, k0 + kchunk - 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool valid = i <= nx - 2 && (!THREE_D || j <= ny - 2);
    // loads of threads past the edge take the last interior column, tile
    // positions past the array its last point: neither feeds a valid cell
    unsigned colb = 8u * (unsigned)((min(i, nx - 2) - 1) + nx * (THREE_D ? min(j, ny - 2) - 1 : 0));
    // threads past the edge store the 0 of an east or north ghost point
    const unsigned outb = 8u * (unsigned)((min(i, nx) - 1) + nx * (THREE_D ? min(j, ny) - 1 : 0));
    const int own = (THREE_D ? (ty + H) * LW : 0) + tx + H;
    auto lev = [&](int kk) { return (size_t)(min(max(kk, 1), nz) - 1) * plane; };
    // element at a 32-bit byte offset from a wave-uniform level plane
    auto at = [&](const double *a, int kk, unsigned byte) {
        return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a + lev(kk)) + byte);
    };
    unsigned off[TS];
#pragma unroll
    for (int s = 0; s < TS; ++s) {
        const int e = min(tid + s * NT, PL - 1), r = e / LW, cc = e - r * LW;
        const int ii = min(i0 - H + cc, nx), jj = THREE_D ? min(j0 - H + r, ny) : 1;
        off[s] = 8u * (unsigned)((ii - 1) + nx * (jj - 1));
    }
    // ghost points next to this item's edge cells are 0
    if (valid) {
        const int ia = i == 4 ? 1 : i, ib = i == nx - 2 ? nx : i;
        const int ja = THREE_D && j == 4 ? 1 : j, jb = THREE_D && j == ny - 2 ? ny : j;
        if (ia < i || ib > i || ja < j || jb > j)
            for (int k = k0; k <= k1; ++k)
                for (int jj = ja; jj <= jb; ++jj)
                    for (int ii = ia; ii <= ib; ++ii) {
                        if (ii == i && jj == j) continue;
                        const size_t id = (size_t)(k - 1) * plane + (size_t)(ii - 1) + (size_t)nx * (jj - 1);
                        ua[id] = 0.0;
                        if (THREE_D) va[id] = 0.0;
                        wa[id] = 0.0;
                    }
    }
    // rings start with levels k0-2..k0
#pragma unroll
    for (int s = 0; s < TS; ++s) {
        const int e = tid + s * NT;
        if (e >= PL) continue;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const int kk = k0 - 2 + n;
            rut[kk & 3][e] = at(ut, kk, off[s]);
            if constexpr (THREE_D) rvt[kk & 3][e] = at(vt, kk, off[s]);
        }
    }
    // own-column windows, levels k-2..k+2
    double zu[5], zv[5], zw[5], zt[5];
#pragma unroll
    for (int n = 0; n < 5; ++n) {
        zu[n] = at(mu, k0 - 2 + n, colb);
        zv[n] = THREE_D ? at(mv, k0 - 2 + n, colb) : 0.0;
        zw[n] = at(mw, k0 - 2 + n, colb);
        zt[n] = at(wt, k0 - 2 + n, colb);
    }
    // thickness of level kk (1 outside the column: never used there)
    auto thick = [&](int kk) { return kk >= 1 && kk <= nz ? dzw[kk - 1] : 1.0; };
    // flux of face kk + 1/2 of the horizontal momenta: the vertical velocity
    // averaged across the line times the momentum weighted with the
    // thicknesses lo, hi of levels kk, kk+1
    auto zflux = [&](double ww, const LevelDiv &d, double lo, double hi, double mlo, double mhi) {
        return ww * d.div(hi * mhi + lo * mlo);
    };
    // advwz_fd: flux and wide flux of w face kk + 1/2, kk < nz (windadv.f90:
    // 1077-1098; the reference writes the top flux as 0.25 (T + T)(M + M), the
    // same product)
    auto wflux = [&](double t0, double t1, double m0, double m1) { return ((t1 + t0) * 0.5) * ((m1 + m0) * 0.5); };
    auto wadvf = [&](int kk, const LevelDiv &d, double lo, double hi, double t0, double t1, double t2, double m0,
                     double m1, double m2) -> double {
        if (kk == nz - 1) {
            const double s = hi + lo;
            if (bc6 == 1) return (0.0 + lo * t0) * (0.0 + lo * m0) / (s * s);
            if (bc6 == 2) return (hi * t1 + lo * t0) * (hi * m1 + lo * m0) / (s * s);
            return 0.0;
        }
        if (kk >= nz || kk < 1) return 0.0;
        return d.div(hi * t2 + lo * t0) * d.div(hi * m2 + lo * m0);
    };
    for (int n = tid; n < k1 - k0 + 3; n += NT) {
        const int kk = k0 - 1 + n;
        const LevelDiv two(thick(kk + 1) + thick(kk)), three(thick(kk - 1) + thick(kk) + thick(kk + 1));
        double *e = lmet + n * NM;
        e[0] = thick(kk);
        e[1] = two.d;
        e[2] = two.r;
        e[3] = three.d;
        e[4] = three.r;
        e[5] = kk >= 1 && kk <= nz ? dz1w[kk - 1] : 0.0;
        e[7] = thick(kk + 1);
        e[6] = kk >= 2 && kk <= nz ? dz1[kk - 2] : 0.0;
    }
    // fluxes of faces k-2..k+1; at the start of the chunk those below k0+1
    // come from memory.  flux(0) is 0, or flux(1) for an 'ope' floor; flux(nz)
    // is 0, or flux(nz-1) for an 'ope' lid.
    double fu[4] = {0.0, 0.0, 0.0, 0.0}, fv[4] = {0.0, 0.0, 0.0, 0.0};
    double wx0 = 0.0, wx1 = 0.0, wy0 = 0.0, wy1 = 0.0;  // wt at (i-1, j) and (i, j-1), levels k, k+1
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const int kk = k0 - 2 + n;  // face kk + 1/2 reads wt at level kk + 1
        const double *wl = wt + lev(kk + 1) + colb / 8u;
        wx0 = wx1;
        wy0 = wy1;
        wx1 = wl[-1];
        wy1 = THREE_D ? wl[-nx] : 0.0;
        if (kk >= 1 && kk < nz) {
            const double lo = dzw[kk - 1], hi = dzw[kk];
            const LevelDiv d(hi + lo);
            fu[n] = zflux(interp4(c, wx1, wl[0], wl[-2], wl[1]), d, lo, hi, zu[n], zu[n + 1]);
            if (THREE_D) fv[n] = zflux(interp4(c, wy1, wl[0], wl[-2 * nx], wl[nx]), d, lo, hi, zv[n], zv[n + 1]);
        }
    }
    if (bc5 == 2 && k0 == 1) {
        fu[1] = fu[2];
        fv[1] = fv[2];
    }
    if (bc5 == 2 && k0 == 2) {
        fu[0] = fu[1];
        fv[0] = fv[1];
    }
    if (bc6 == 2 && k0 == nz) {
        fu[2] = fu[1];
        fv[2] = fv[1];
    }
    // flux(k-1), wide fluxes of k-1 and k-2 of w
    double wf1 = k0 > 1 ? wflux(zt[1], zt[2], zw[1], zw[2]) : 0.0;
    const double ha = thick(k0 - 2), hb = thick(k0 - 1), hc = thick(k0);
    double wa1 = wadvf(k0 - 1, LevelDiv(hc + hb), hb, hc, zt[1], zt[2], zt[3], zw[1], zw[2], zw[3]);
    double wa2 = wadvf(k0 - 2, LevelDiv(hb + ha), ha, hb, zt[0], zt[1], zt[2], zw[0], zw[1], zw[2]);
    if (bc5 == 2 && k0 == 2) wa2 = wf1;
    const double dz1w1 = dz1w[0];
    // byte offsets of levels k+1..k+3 (the last level beyond it)
    const size_t pb = plane * sizeof(double), last = lev(nz) * sizeof(double);
    size_t o1 = lev(k0) * sizeof(double), o2 = lev(k0 + 1) * sizeof(double), o3 = lev(k0 + 2) * sizeof(double);
    // slot values of the next level: momenta at k, ut and vt at k+1, wt at k+2
    double nm[3][TS], nu[TS], nv[TS], nw[TS];
    auto ld = [&](const double *a, size_t o, unsigned byte) {
        return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a) + o + byte);
    };
    auto fetch = [&]() {
#pragma unroll
        for (int s = 0; s < TS; ++s) {
            nu[s] = ld(ut, o2, off[s]);
            if (THREE_D) nv[s] = ld(vt, o2, off[s]);
            nm[0][s] = ld(mu, o1, off[s]);
            if (THREE_D) nm[1][s] = ld(mv, o1, off[s]);
            nm[2][s] = ld(mw, o1, off[s]);
            nw[s] = ld(wt, o3, off[s]);
        }
    };
    fetch();
    auto up = [&]() {
        o1 = o2;
        o2 = o3;
        o3 = min(o3 + pb, last);
    };
    up();
    // The first level's operands are waited for here: the waits inside the loop
    // then count what a level itself has in flight (its stores may stay), not
    // the fewer requests of the way into it.
#pragma unroll
    for (int s = 0; s < TS; ++s) {
        settle(nu[s]);
        settle(nm[0][s]);
        settle(nm[2][s]);
        settle(nw[s]);
        if constexpr (THREE_D) {
            settle(nv[s]);
            settle(nm[1][s]);
        }
    }
    // the own-column windows enter a level one step behind, with its top value
    // in cu..ct: the shift then waits for the loads after the first barrier
    double cu = zu[4], cv = zv[4], cw = zw[4], ct = zt[4];
#pragma unroll
    for (int n = 4; n > 0; --n) {
        zu[n] = zu[n - 1];
        zv[n] = zv[n - 1];
        zw[n] = zw[n - 1];
        zt[n] = zt[n - 1];
    }
#pragma unroll 1
    for (int k = k0; k <= k1; ++k) {
        // the offsets are opaque per level: otherwise every array's 64-bit
        // address is hoisted out of the loop into registers of its own
#pragma unroll
        for (int s = 0; s < TS; ++s) asm volatile("" : "+v"(off[s]));
        asm volatile("" : "+v"(colb));
#pragma unroll
        for (int s = 0; s < TS; ++s) {
            const int e = tid + s * NT;
            if (e >= PL) continue;
            lmu[e] = nm[0][s];
            lmw[e] = nm[2][s];
            lw[e] = nw[s];
            rut[(k + 1) & 3][e] = nu[s];
            if constexpr (THREE_D) {
                lmv[e] = nm[1][s];
                rvt[(k + 1) & 3][e] = nv[s];
            }
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            zu[n] = zu[n + 1];
            zv[n] = zv[n + 1];
            zw[n] = zw[n + 1];
            zt[n] = zt[n + 1];
        }
        zu[4] = cu;
        zv[4] = cv;
        zw[4] = cw;
        zt[4] = ct;
        // averages of the advecting components, once per point
        const double *lut = rut[k & 3], *lvt = rvt[THREE_D ? k & 3 : 0];
        const double *lub = rut[(k - 1) & 3], *lvb = rvt[THREE_D ? (k - 1) & 3 : 0];
        {
            // the w levels 2 and nz take the two-point average
            const bool two = k == 2 || k == nz;
            auto across = [&](double n1, double n2, double f1, double f2) {
                const double far = c.c2c * (f1 + f2) * 0.5;
                return (two ? 1.0 : c.c1c) * (n1 + n2) * 0.5 - (two ? 0.0 : far);
            };
            const double *u1 = rut[(k + 1) & 3], *u2 = rut[(k - 2) & 3];
            const double *v1 = rvt[THREE_D ? (k + 1) & 3 : 0], *v2 = rvt[THREE_D ? (k - 2) & 3 : 0];
            // point s of this thread in both lists: all reads, then all
            // arithmetic, then the writes, so that one wait serves them (a
            // wave of short lists is the last to reach the barrier)
            auto point = [&](int s) {
                const int e = tid + s * NT, eu = min(e, UW * TY - 1), ev = min(e, NVX - 1);
                const int ru = eu / UW, o = (THREE_D ? ru + H : 0) * LW + eu - ru * UW + 1;
                const int rv = ev / TX, q = (rv + 1) * LW + ev - rv * TX + H;
                const double a0 = lut[o], a1 = lub[o], a2 = u1[o], a3 = u2[o];
                double b0 = 0.0, b1 = 0.0, b2 = 0.0, p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0, t0 = 0.0, t1 = 0.0, t2 = 0.0;
                if constexpr (THREE_D) {
                    b0 = lut[o - LW];
                    b1 = lut[o - 2 * LW];
                    b2 = lut[o + LW];
                    p0 = lvt[q];
                    p1 = lvb[q];
                    p2 = v1[q];
                    p3 = v2[q];
                    t0 = lvt[q - 1];
                    t1 = lvt[q - 2];
                    t2 = lvt[q + 1];
                }
                const double uu = across(a0, a1, a2, a3), uy = interp4(c, b0, a0, b1, b2);
                const double vv = across(p0, p1, p2, p3), vx = interp4(c, t0, p0, t1, t2);
                if (e < UW * TY) {
                    luu[e] = uu;
                    if constexpr (THREE_D) luy[e] = uy;
                }
                if constexpr (THREE_D) {
                    if (e < NVX) {
                        lvv[e] = vv;
                        lvx[e] = vx;
                    }
                }
            };
            point(0);
            constexpr int REST = (THREE_D ? std::max(NVX, UW * TY) : UW * TY) - NT;
            static_assert(REST <= NT, "two points per thread");
            if (REST > 0 && (tid & ~63) < REST) point(1);
        }
        __syncthreads();
        const size_t kb = (size_t)(k - 1) * plane;
        auto put = [&](double *o, double v) {
            *reinterpret_cast<double *>(reinterpret_cast<char *>(o + kb) + outb) = valid ? v : 0.0;
        };
        // vertical fluxes of face k+1 (+1/2), wt at level k+2
        const LevelZ lz(k, nz, bc5, bc6);
        const double *met = lmet + (k - k0) * NM;  // level k-1
        const LevelDiv pp(met[2 * NM + 1], met[2 * NM + 2]);
        const double h2 = met[2 * NM], h3 = met[2 * NM + 7];
        const double *wl = lw + own;
        const double wx2 = wl[-1], wy2 = THREE_D ? wl[-LW] : 0.0;
        fu[3] = zflux(interp4(c, wx2, wl[0], wl[-2], wl[1]), pp, h2, h3, zu[3], zu[4]);
        if (THREE_D) fv[3] = zflux(interp4(c, wy2, wl[0], wl[-2 * LW], wl[LW]), pp, h2, h3, zv[3], zv[4]);
        if (k + 1 >= nz) {
            fu[3] = bc6 == 2 ? fu[2] : 0.0;
            fv[3] = bc6 == 2 ? fv[2] : 0.0;
        }
        settle(fu[3]);
        settle(fv[3]);
        const LevelDiv d3(met[NM + 3], met[NM + 4]);
        const double dz1wk = met[NM + 5];
        // values along x and y through this cell, whose own value is known
        auto alongx = [&](const double *l, double mid, double *m) {
#pragma unroll
            for (int n = 0; n < 5; ++n) m[n] = n == 2 ? mid : l[own + n - 2];
        };
        auto alongy = [&](const double *l, double mid, double *m) {
#pragma unroll
            for (int n = 0; n < 5; ++n) m[n] = n == 2 ? mid : l[own + (n - 2) * LW];
        };
        // the directions of one component in the order of ntime
        auto sum = [&](auto x, auto y, auto z) {
            double t = EVEN ? x(0.0) : z(0.0);
            settle(t);
            if constexpr (THREE_D) {
                t = y(t);
                settle(t);
            }
            t = EVEN ? z(t) : x(t);
            settle(t);
            return t;
        };
        const double u0 = lut[own], v0 = THREE_D ? lvt[own] : 0.0;
        // ---- u (uadv_fd, windadv.f90:82-220)
        const double ru = sum(
                    [&](double t) {
                        double m[5], u[5];
                        alongx(lmu, zu[2], m);
                        alongx(lut, u0, u);
                        return self_line<VISC>(t, m, u, c.dx1, c.dx2, c);
                    },
                    [&](double t) {
                        double m[5], vv[4];
                        alongy(lmu, zu[2], m);
#pragma unroll
                        for (int n = 0; n < 4; ++n) vv[n] = lvx[(ty + n) * TX + tx];
                        const double *v = lvt + own;
                        return cross_line<VISC>(t, m, vv, VISC ? v[-1] + v0 + v[LW - 1] + v[LW] : 0.0, c.dy1, c.dy3, c);
                    },
                    [&](double t) {
                        const double mu = 0.25 * fabs(wx0 + zt[2] + wx1 + zt[3]) * dz1wk;
                        return lz.template add<VISC>(t, fu[2] - fu[1], fu[3] - fu[0], c.c1c, c.c2c,
                                                     k == 2 ? dz1w1 : dz1wk, d3, mu, zu);
                    });
        // ---- v (vadv_fd, windadv.f90:223-357)
        double rv = 0.0;
        if constexpr (THREE_D)
            rv = sum(
                        [&](double t) {
                            double m[5], vv[4];
                            alongx(lmv, zv[2], m);
#pragma unroll
                            for (int n = 0; n < 4; ++n) vv[n] = luy[ty * UW + tx + n];
                            const double *u = lut + own;
                            return cross_line<VISC>(t, m, vv, VISC ? u[-LW] + u0 + u[1 - LW] + u[1] : 0.0, c.dx1,
                                                    c.dx3, c);
                        },
                        [&](double t) {
                            double m[5], v[5];
                            alongy(lmv, zv[2], m);
                            alongy(lvt, v0, v);
                            return self_line<VISC>(t, m, v, c.dy1, c.dy2, c);
                        },
                        [&](double t) {
                            const double mu = 0.25 * fabs(wy0 + zt[2] + wy1 + zt[3]) * dz1wk;
                            return lz.template add<VISC>(t, fv[2] - fv[1], fv[3] - fv[0], c.c1c, c.c2c, dz1wk, d3, mu,
                                                         zv);
                        });
        // requests for the next level
        if (k < k1) {
            fetch();
            cu = ld(mu, o3, colb);
            cv = THREE_D ? ld(mv, o3, colb) : 0.0;
            cw = ld(mw, o3, colb);
            ct = ld(wt, o3, colb);
            up();
        }
        // ---- w (wadv_fd, windadv.f90:360-492): levels 2..nz
        double wf0 = wflux(zt[2], zt[3], zw[2], zw[3]);
        if (k == nz) wf0 = bc6 == 2 ? wf1 : 0.0;
        const double wa0 = wadvf(k, LevelDiv(met[NM + 1], met[NM + 2]), met[NM], h2, zt[2], zt[3], zt[4], zw[2], zw[3], zw[4]);
        const double rw = sum(
            [&](double t) {
                double m[5], vv[4];
                alongx(lmw, zw[2], m);
#pragma unroll
                for (int n = 0; n < 4; ++n) vv[n] = luu[ty * UW + tx + n];
                return cross_line<VISC>(t, m, vv, VISC ? u0 + lub[own] + lut[own + 1] + lub[own + 1] : 0.0, c.dx1,
                                        c.dx3, c);
            },
            [&](double t) {
                double m[5], vv[4];
                alongy(lmw, zw[2], m);
#pragma unroll
                for (int n = 0; n < 4; ++n) vv[n] = lvv[(ty + n) * TX + tx];
                return cross_line<VISC>(t, m, vv, VISC ? v0 + lvb[own] + lvt[own + LW] + lvb[own + LW] : 0.0, c.dy1,
                                        c.dy3, c);
            },
            [&](double t) {
                const double d1 = met[NM + 6];
                return lz.template add<VISC>(t, wf0 - wf1, wa0 - wa2, c.c1s, c.c2s, d1, LevelDiv(met[1], met[2]),
                                             fabs(zt[2]) * d1, zw);
            });
        // stored after the requests, and by every thread: the next level then
        // waits for its operands without waiting for these stores
        put(ua, ru);
        if (THREE_D) put(va, rv);
        put(wa, k >= 2 ? rw : 0.0);
        // what level k+1 takes over
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            fu[n] = fu[n + 1];
            fv[n] = fv[n + 1];
        }
        wx0 = wx1;
        wy0 = wy1;
        wx1 = wx2;
        wy1 = wy2;
        wf1 = wf0;
        wa2 = k == 1 && bc5 == 2 ? wf0 : wa1;  // advf(0) of an 'ope' floor is flux(1)
        wa1 = wa0;
        __syncthreads();  // every read of this level's tiles is done
    }
}

MomCoefs mom_coefs(const GridDev &g, int mom_ord)
{
    MomCoefs c;
    if (mom_ord == 4) {
        c.c1s = 4.0 / 3.0; c.c2s = 1.0 / 3.0;
        c.c1c = 9.0 / 8.0; c.c2c = 1.0 / 8.0;
    } else {
        c.c1s = 1.0; c.c2s = 0.0;
        c.c1c = 1.0; c.c2c = 0.0;
    }
    c.dx1 = 1.0 / g.dx;
    c.dx2 = 1.0 / (2.0 * g.dx);
    c.dx3 = 1.0 / (3.0 * g.dx);
    c.dy1 = 1.0 / g.dy;
    c.dy2 = 1.0 / (2.0 * g.dy);
    c.dy3 = 1.0 / (3.0 * g.dy);
    return c;
}

template <int TX, int TY, bool VISC, bool EVEN>
hipError_t launch_tile(const GridDev &g, const MomCoefs &c, const double *mu, const double *mv, const double *mw,
                       const double *ut, const double *vt, const double *wt, double *ua, double *va, double *wa,
                       hipStream_t s)
{
    const int ntx = (g.nx - 5 + TX - 1) / TX, nty = TY > 1 ? (g.ny - 5 + TY - 1) / TY : 1;
    // Two rounds of resident items fill the device and overlap the start of one
    // item with the levels of others: 16-level items take 280 us at 256x256x128
    // against 333 us for 43 levels (one round exactly), 1-level items 22 us at
    // 64x64x48 against 49 us for 8 levels.
    const int kchunk = levels_per_item(g.nz, (long)ntx * nty, 2 * MOM_GROUPS, MOM_LEVELS);
    const int nwork = ntx * nty * ((g.nz + kchunk - 1) / kchunk);
    hipLaunchKernelGGL((momentum_march_kernel<TX, TY, VISC, EVEN>), dim3(nwork), dim3(TX * TY), 0, s, g, c, mu, mv, mw, ut, vt, wt,
                       g.zm.dzw, g.zm.dz1w, g.zm.dz1, ua, va, wa, kchunk, ntx, nwork);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_momentum_fp64(const GridDev &g, int mom_ord, int lavisc, int ntime, const double *mu,
                                const double *mv, const double *mw, const double *ut, const double *vt,
                                const double *wt, double *ua, double *va, double *wa, hipStream_t s)
{
    const MomCoefs c = mom_coefs(g, mom_ord);
    auto go = [&](auto visc, auto even) {
        constexpr bool V = decltype(visc)::value, E = decltype(even)::value;
        return g.ny > 1 ? launch_tile<32, 8, V, E>(g, c, mu, mv, mw, ut, vt, wt, ua, va, wa, s)
                        : launch_tile<64, 1, V, E>(g, c, mu, mv, mw, ut, vt, wt, ua, va, wa, s);
    };
    using std::false_type;
    using std::true_type;
    if (ntime % 2 == 0) return lavisc ? go(true_type{}, true_type{}) : go(false_type{}, true_type{});
    return lavisc ? go(true_type{}, false_type{}) : go(false_type{}, false_type{});
}

}  // namespace mimadv
