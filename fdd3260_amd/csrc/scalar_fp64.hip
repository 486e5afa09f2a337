// scalar_fp64.hip -- plain per-field FP64 scalar advection on gfx950: the PPM
// kernel and the scheme dispatch (the other schemes run on the kernels of
// weno_march.hip).
//
// One launch computes the fused x+y+z flux divergence of one field
// (advection_x/y/z of src/TOOLS/advection.f90:556-798 for all three
// directions) and applies one of the epilogues of ScalarArgs: accumulate
// into a tendency, overwrite it, or a full Heun / Shu-Osher stage update
// with the periodic ghost images written in the same pass (so no separate
// statebc/qnbc_p4 sweep is needed between stages).
//
// This file is compiled with -ffp-contract=off: the arithmetic follows the
// reference operation order and matches the CPU restatement bit for bit.
#include "mimadv_internal.hpp"

namespace mimadv {

namespace {

// One work item: a TX x TY column tile marched up a chunk of levels.
//
// What bounds it: vector issue.  A cell record (limiter_ppm and the CW84
// averages Flux_r, Flux_l) is about 130 instructions, so each is formed once:
// per level the plane tile with a 3-cell halo and the face velocities go
// through LDS, the x records of the cells i0-1..i0+TX of each row and the y
// records of j0-1..j0+TY of each column are formed by a flattened loop over
// the group, and the z record of level k+1 is formed once by its column's
// thread and carried up (its differences, gammas and face value with it).
// 3.3 records per cell; a chunk above the floor first forms two z records.
// 128 VGPRs (a dozen loop-invariant offsets spill) give four groups per CU.
//
// Measured against one group per tile and level with 5.5 records per cell and
// full divisions in the limiter (1670 vector instructions per cell, now 760):
// 256x256x128 430 -> 280 us, 139x117x75 96 -> 63 us, 128x128 (2D) 11.6 -> 10.3
// us.  32x8 tiles take 314 us, 144 VGPRs without spills (three groups) 300 us.
// (228 us per field at 256x256x128 since the level metrics are scalar loads and
// two fields share a launch.)
template <int TX, int TY>
__global__ __launch_bounds__(TX *TY) __attribute__((amdgpu_waves_per_eu(4, 8))) void ppm_march_kernel(
    GridDev g, SchemeParams sp, ScalarList l, int kchunk, int ntx)
{
    const ScalarArgs a = l.field(blockIdx.y);
    constexpr bool THREE_D = TY > 1;
    constexpr int NT = TX * TY, H = 3;
    constexpr int LW = TX + 2 * H, LH = THREE_D ? TY + 2 * H : 1, PL = LW * LH;
    constexpr int NXR = TY * (TX + 2), NYR = THREE_D ? (TY + 2) * TX : 0, NR = NXR + NYR;
    // velocities: u(i0-1..i0+TX+1) of each row, v(j0-1..j0+TY+1) of each column
    constexpr int UW = TX + 3, NU = TY * UW, NVEL = NU + (THREE_D ? (TY + 3) * TX : 0);
    constexpr int TS = (PL + NT - 1) / NT, VS = (NVEL + NT - 1) / NT, RS = (NR + NT - 1) / NT;
    __shared__ double tile[PL];
    __shared__ double vel[NVEL];
    __shared__ double rfr[NR], rfl[NR];

    const int nx = g.nx, ny = g.ny, nz = g.nz, mx = nx - 5, my = ny - 5;
    const size_t plane = (size_t)nx * ny;
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int nchunk = (nz + kchunk - 1) / kchunk;
    const int tile_id = blockIdx.x / nchunk, kc = blockIdx.x - tile_id * nchunk;
    const int i0 = 4 + (tile_id % ntx) * TX, j0 = THREE_D ? 4 + (tile_id / ntx) * TY : 1;
    const int k0 = 1 + kc * kchunk, k1 = min(nz, k0 + kchunk - 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool valid = i <= nx - 2 && (!THREE_D || j <= ny - 2);
    unsigned col = 8u * (unsigned)((min(i, nx - 2) - 1) + nx * (THREE_D ? min(j, ny - 2) - 1 : 0));
    const double dx1 = 1.0 / g.dx, dy1 = 1.0 / g.dy, dt0 = sp.dt0;
    const bool adv = a.adv != 0, xdir = (a.dirmask & 1) != 0, ydir = THREE_D && (a.dirmask & 2),
               zdir = (a.dirmask & 4) != 0;
    const int bc5 = g.bcl[4], bc6 = g.bcl[5];
    const double bc51 = bc5 == 0 ? 1.0 : 0.0, bc61 = bc6 == 0 ? 1.0 : 0.0;
    const auto dz1w = table(g.zm.dz1w), dz1 = table(g.zm.dz1), ppmc = table(g.zm.ppmc);
    const bool accum = a.epi == EPI_ACCUM, heun = a.epi == EPI_HEUN, so = a.epi == EPI_SO;
    const bool need_tend = heun && a.b_lm != 0.0;
    // the array the epilogue starts from: the tendency or the step-start state
    const double *base = accum ? a.xs : (heun || so ? a.q0 : nullptr);
    // positions past the array (padding of a partial tile) read a periodic
    // image that feeds no interior cell
    auto img = [](int x, int n, int m) { return x > n ? (x - 4) % m + 4 : x; };
    unsigned toff[TS], voff[VS];
#pragma unroll
    for (int s = 0; s < TS; ++s) {
        const int e = min(tid + s * NT, PL - 1), r = e / LW, c = e - r * LW;
        toff[s] = 8u * (unsigned)((img(i0 - H + c, nx, mx) - 1) + (THREE_D ? nx * (img(j0 - H + r, ny, my) - 1) : 0));
    }
#pragma unroll
    for (int s = 0; s < VS; ++s) {
        const int e = min(tid + s * NT, NVEL - 1);
        if (e < NU) {
            const int r = e / UW, c = e - r * UW;
            voff[s] = 8u * (unsigned)((img(i0 - 1 + c, nx, mx) - 1) + (THREE_D ? nx * (img(j0 + r, ny, my) - 1) : 0));
        } else {
            const int e2 = e - NU, r = e2 / TX, c = e2 - r * TX;
            voff[s] = 8u * (unsigned)((img(i0 + c, nx, mx) - 1) + nx * (img(j0 - 1 + r, ny, my) - 1));
        }
    }
    // record 3 or n-1 of a line lies in this item
    const bool edge = i0 == 4 || i0 + TX > nx - 2 || (THREE_D && (j0 == 4 || j0 + TY > ny - 2));

    // element at a 32-bit byte offset from a wave-uniform level plane
    auto at = [&](const double *p, unsigned byte) {
        return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(p) + byte);
    };
    auto put = [&](double *p, unsigned byte, double v) {
        *reinterpret_cast<double *>(reinterpret_cast<char *>(p) + byte) = v;
    };
    auto Q = [&](int kk) { return at(a.q + (size_t)(kk - 1) * plane, col); };
    auto W = [&](int kk) { return kk >= 1 && kk <= nz ? at(a.w + (size_t)(kk - 1) * plane, col) : 0.0; };
    // difference D(m) = Q(m+1) - Q(m); D(0), D(-1) and D(nz) are what the
    // reference puts beyond a periodic (else closed) floor and lid, `near` =
    // D(nz-1) the neighbour of the lid
    auto below = [&](int m) { return bc51 * (m == 0 ? Q(nz - 4) - Q(nz - 5) : Q(nz - 5) - Q(nz - 6)); };
    auto lid = [&](double near) { return bc61 * (Q(6) - Q(5)) + (1.0 - bc61) * near; };

    // z state of iteration k, which forms the record of level c = k+1
    const int kstart = zdir ? max(k0 - 2, 0) : k0;
    double qm = 0.0, qc = 0.0, qp = 0.0;     // Q(c-1), Q(c), Q(c+1)
    double dm2 = 0.0, dm1 = 0.0, d0 = 0.0;   // D(c-2), D(c-1), D(c)
    double gm = 0.0, g0 = 0.0;               // ppm_gamma of (D(c-1), D(c-2)), (D(c), D(c-1))
    double xlo = 0.0;                        // left face value of c
    double wc = 0.0;                         // W(c)
    double frk = 0.0, fzb = 0.0;             // Flux_r of level k, flux of face k-1
    double qn = 0.0, wn = 0.0;               // Q(c+2), W(c+1), requested one level ahead
    if (zdir) {
        const int c = kstart + 1;
        qc = Q(c);
        qp = c < nz ? Q(c + 1) : 0.0;
        wc = W(c);
        d0 = c < nz ? qp - qc : 0.0;
        if (c == 1) {
            qm = qp;  // the reference passes x(2) as the lower neighbour
            dm1 = below(0);
            dm2 = below(-1);
            xlo = qc - 0.5 * d0;
        } else {
            qm = Q(c - 1);
            dm1 = qc - qm;
            dm2 = c == 2 ? below(0) : qm - Q(c - 2);
            if (c < nz) xlo = ppm_zxplus(c - 1, nz, ppmc, qm, dm2, dm1, d0);
        }
        gm = ppm_gamma(dm1, dm2);
        g0 = ppm_gamma(d0, dm1);
        qn = c + 2 <= nz ? Q(c + 2) : 0.0;
        wn = W(c + 1);
    } else {
        qm = Q(k0);
    }

    // operands of level k, requested one level ahead
    double tv[TS], vv[VS], basev = 0.0, tdv = 0.0;
    auto fetch = [&](int k) {
        const size_t kb = (size_t)(k - 1) * plane;
        const double *qk = a.q + kb, *uk = a.u + kb, *vk = a.v + kb;
#pragma unroll
        for (int s = 0; s < TS; ++s) tv[s] = at(qk, toff[s]);
#pragma unroll
        for (int s = 0; s < VS; ++s) {
            const bool isu = tid + s * NT < NU;
            vv[s] = 0.0;
            if (isu ? xdir : ydir) vv[s] = isu ? at(uk, voff[s]) : at(vk, voff[s]);
        }
        if (base) basev = at(base + kb, col);
        if (need_tend) tdv = at(a.tend + kb, col);
    };
    fetch(k0);
#pragma unroll 1
    for (int k = kstart; k <= k1; ++k) {
        // the offsets are opaque per level: otherwise every array's 64-bit
        // address is hoisted out of the loop into registers of its own
#pragma unroll
        for (int s = 0; s < TS; ++s) asm volatile("" : "+v"(toff[s]));
#pragma unroll
        for (int s = 0; s < VS; ++s) asm volatile("" : "+v"(voff[s]));
        asm volatile("" : "+v"(col));
        double fzt = 0.0, wk = 0.0;  // flux of face k, W(k+1)
        if (zdir) {
            const int c = k + 1;
            wk = wc;
            double fr = 0.0, fl = 0.0, dp = 0.0, gp = 0.0, xhi = 0.0;
            if (c < nz) {
                dp = c + 1 < nz ? qn - qp : lid(d0);
                gp = ppm_gamma(dp, d0);
                xhi = ppm_zxplus(c, nz, ppmc, qc, dm1, d0, dp);
                const double mup = fabs(wn) * dt0 * dz1[c - 1], muc = fabs(wc) * dt0 * dz1[c - 1];
                const PPMRec r = ppm_cell(sp.ppm_limiter, qc, qp, qm, xhi, xlo, d0, dp, dm1, dm2, g0, gp, gm, mup, muc);
                fr = r.fr;
                fl = r.fl;
            } else if (c == nz) {
                // Flux_l of the top level (advq_ppm.f90:411-414)
                const double muc = fabs(wc) * dt0 * dz1[nz - 1];
                fl = qc + 0.5 * dm1 * (1.0 - muc);
            }
            if (k >= 1 && k < nz) fzt = ppm_faceflux(frk, fl, wc);
            // to level k+1
            frk = fr;
            qm = qc;
            qc = qp;
            qp = qn;
            dm2 = dm1;
            dm1 = d0;
            d0 = dp;
            gm = g0;
            g0 = gp;
            xlo = xhi;
            wc = wn;
            if (k < k1) {
                qn = c + 3 <= nz ? Q(c + 3) : 0.0;
                wn = W(c + 2);
            }
        }
        if (k < k0) {
            fzb = fzt;
            continue;
        }
        // the z record is finished here (its temporaries do not fit the
        // registers beside the rest)
        settle(fzt);
        settle(frk);
        const size_t kb = (size_t)(k - 1) * plane;
#pragma unroll
        for (int s = 0; s < TS; ++s)
            if (tid + s * NT < PL) tile[tid + s * NT] = tv[s];
#pragma unroll
        for (int s = 0; s < VS; ++s)
            if (tid + s * NT < NVEL) vel[tid + s * NT] = vv[s];
        const double basec = basev, tdc = tdv;
        __syncthreads();
        if (k < k1) fetch(k + 1);
        // one record at a time: ppm_cell is register-hungry
#pragma unroll 1
        for (int s = 0; s < RS; ++s) {
            const int e = tid + s * NT;
            if (e >= NR) break;
            int b, st, c, n;
            double u0, u1, d1;
            if (e < NXR) {
                if (!xdir) continue;
                const int r = e / (TX + 2), cc = e - r * (TX + 2);
                b = (THREE_D ? r + H : 0) * LW + cc + 2;
                st = 1;
                c = i0 - 1 + cc;
                n = nx;
                u0 = vel[r * UW + cc];
                u1 = vel[r * UW + cc + 1];
                d1 = dx1;
            } else {
                if (!ydir) break;
                const int e2 = e - NXR, r = e2 / TX, cc = e2 - r * TX;
                b = (r + 2) * LW + cc + H;
                st = LW;
                c = j0 - 1 + r;
                n = ny;
                u0 = vel[NU + r * TX + cc];
                u1 = vel[NU + (r + 1) * TX + cc];
                d1 = dy1;
            }
            const double mup = fabs(u1) * dt0 * d1, muc = fabs(u0) * dt0 * d1;
            const double m2 = tile[b - 2 * st], m1 = tile[b - st], x0 = tile[b], p1 = tile[b + st], p2 = tile[b + 2 * st];
            const PPMRec r = edge ? ppm_hcell<true>(c, n, sp, m2, m1, x0, p1, p2, mup, muc)
                                  : ppm_hcell<false>(c, n, sp, m2, m1, x0, p1, p2, mup, muc);
            rfr[e] = r.fr;
            rfl[e] = r.fl;
        }
        // what the cell takes from the tile and the velocities is read here: the
        // next level's values go there as soon as the barrier is passed
        const double qcell = tile[(THREE_D ? ty + H : 0) * LW + tx + H];
        const double ui = vel[ty * UW + tx + 1], uip = vel[ty * UW + tx + 2];
        double vj = 0.0, vjp = 0.0;
        if constexpr (THREE_D) {
            vj = vel[NU + (ty + 1) * TX + tx];
            vjp = vel[NU + (ty + 2) * TX + tx];
        }
        __syncthreads();
        if (valid) {
            double X = 0.0, Y = 0.0, Z = 0.0;
            if (xdir) {
                // ppm_h (advq_ppm.f90:136-163) on the records of cells i-1, i, i+1
                const int e = ty * (TX + 2) + tx;
                double fr_i = rfr[e + 1], fl_ip = rfl[e + 2];
                if (g.bcl[1] != 0 && i == nx - 2) {
                    fr_i = rfl[e + 1];  // Flux_r(ii2) = Flux_l(ii2)
                    fl_ip = rfr[e];     // Flux_l(ii2+1) = Flux_r(ii2-1)
                }
                const double flux_old = ppm_faceflux(rfr[e], rfl[e + 1], ui);
                X = (ppm_faceflux(fr_i, fl_ip, uip) - flux_old) * dx1;
                if (adv) X = X - qcell * (uip - ui) * dx1;
            }
            if (ydir) {
                const int e = NXR + ty * TX + tx;
                double fr_j = rfr[e + TX], fl_jp = rfl[e + 2 * TX];
                if (g.bcl[3] != 0 && j == ny - 2) {
                    fr_j = rfl[e + TX];
                    fl_jp = rfr[e];
                }
                const double flux_old = ppm_faceflux(rfr[e], rfl[e + TX], vj);
                Y = (ppm_faceflux(fr_j, fl_jp, vjp) - flux_old) * dy1;
                if (adv) Y = Y - qcell * (vjp - vj) * dy1;
            }
            if (zdir) {
                // no-flux 'nnf' floor/lid, zero z tendency at other ends
                if (k >= 2 && k < nz) {
                    Z = (fzt - fzb) * dz1w[k - 1];
                    if (adv) Z = Z - qcell * (wk - W(k)) * dz1w[k - 1];
                } else if (k == 1 && bc5 == 1) {
                    Z = 0.0 + (fzt - 0.0) * dz1w[0];
                    if (adv) Z = Z - qcell * (wk - 0.0) * dz1w[0];
                } else if (k == nz && bc6 == 1) {
                    Z = 0.0 + (0.0 - fzb) * dz1w[nz - 1];
                    if (adv) Z = Z - qcell * (0.0 - W(nz)) * dz1w[nz - 1];
                }
            }
            double r = accum ? basec : 0.0;
            if (xdir) r = r - X;
            if (ydir) r = r - Y;
            if (zdir) r = r - Z;
            if (accum || a.epi == EPI_OVERWRITE) {
                put(a.xs + kb, col, r);
            } else {
                double q;
                if (heun) {
                    const double T = need_tend ? r + a.b_lm * tdc : r + 0.0;
                    put(a.tend + kb, col, T);
                    q = basec + a.adt * T;
                } else {
                    q = a.c0 * basec + a.c1 * (qcell + a.dt * r);
                }
                put(a.qn + kb, col, q);
                if (a.fill) {
                    // periodic images (qnbc_p4, bc.f90:409-414 and :431-436)
                    int ix = 0, jy = 0;
                    if (i >= nx - 4) ix = i - mx;
                    else if (i <= 5) ix = i + mx;
                    if (THREE_D) {
                        if (j >= ny - 4) jy = j - my;
                        else if (j <= 5) jy = j + my;
                    }
                    double *qo = a.qn + kb;
                    if (ix) qo[(size_t)(ix - 1) + (size_t)nx * (j - 1)] = q;
                    if (jy) {
                        qo[(size_t)(i - 1) + (size_t)nx * (jy - 1)] = q;
                        if (ix) qo[(size_t)(ix - 1) + (size_t)nx * (jy - 1)] = q;
                    }
                }
            }
        }
        fzb = fzt;
    }
}

template <int TX, int TY>
hipError_t launch_ppm(const GridDev &g, const SchemeParams &sp, const ScalarList &a, int nf, int per_cu, hipStream_t s)
{
    const int ntx = (g.nx - 5 + TX - 1) / TX, nty = TY > 1 ? (g.ny - 5 + TY - 1) / TY : 1;
    // a chunk's start costs about one level; sixteen levels at most (longer
    // ones lose the planes of the level above from L2: 456 -> 537 us for two
    // fields at 256x256x128 with 25).  At most as many items as fit one round
    // -> this rule, Heun step: 300x200x100 474 -> 422 us, 190x131x75 (two
    // fields) 349 -> 300 us.
    const int kchunk = levels_by_rounds(g.nz, (long)ntx * nty * nf, per_cu, 1, 16);
    const int items = ntx * nty * ((g.nz + kchunk - 1) / kchunk);
    hipLaunchKernelGGL((ppm_march_kernel<TX, TY>), dim3(items, nf), dim3(TX * TY), 0, s, g, sp, a, kchunk, ntx);
    return hipGetLastError();
}

hipError_t launch_list(const GridDev &g, const SchemeParams &sp, const ScalarList &a, int nf, hipStream_t s)
{
    switch (sp.scheme) {
    case 1: return g.ny > 1 ? launch_ppm<16, 16>(g, sp, a, nf, 4, s) : launch_ppm<64, 1>(g, sp, a, nf, 16, s);
    case 0: case 2: case 3: case 4: case 5: case 6: case 7: return launch_march(g, sp, a, nf, s);
    default: return hipErrorInvalidValue;
    }
}

// Whether what field a writes overlaps nothing that field b reads or writes.
bool writes_apart(const ScalarArgs &a, const ScalarArgs &b, size_t n)
{
    for (const double *w : {a.xs, a.tend, a.qn})
        for (const double *r : {b.q, b.u, b.v, b.w, b.q0, (const double *)b.xs, (const double *)b.tend,
                                (const double *)b.qn}) {
            const uintptr_t p = (uintptr_t)w, q = (uintptr_t)r;
            if (w && r && (p < q ? q - p : p - q) < n * sizeof(double)) return false;
        }
    return true;
}

}  // namespace

// One launch for several fields: a launch per field ends with a round that is
// not full, and the next starts behind it.  SSP-RK3 step of two WENO5 fields
// at 139x117x75 411 -> 376 us, four MUSCL tendencies at 190x131x75 173 -> 150
// us, two PPM tendencies at 256x256x128 484 -> 454 us, Heun step of two 'weno'
// fields there 646 -> 620 us.
hipError_t launch_scalar_fp64(const GridDev &g, const SchemeParams &sp, const ScalarArgs *a, int nf, hipStream_t s)
{
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    for (int f0 = 0; f0 < nf;) {
        ScalarList l = {};
        l.all = a[f0];
        // a component that no direction of the call uses may be missing; the
        // kernels load all of them
        for (const double **c : {&l.all.u, &l.all.v, &l.all.w})
            if (!*c) *c = a[f0].q;
        l.set(0, a[f0]);
        int n1 = 1;
        for (bool ok = true; ok && n1 < SCALAR_FIELDS && f0 + n1 < nf; n1 += ok) {
            const ScalarArgs &b = a[f0 + n1];
            for (int h = f0; h < f0 + n1; ++h) ok = ok && writes_apart(b, a[h], n) && writes_apart(a[h], b, n);
            l.set(n1, b);
        }
        const hipError_t e = launch_list(g, sp, l, n1, s);
        if (e != hipSuccess) return e;
        f0 += n1;
    }
    return hipSuccess;
}

std::vector<double> ppm_coefficients(int nz, const double *dz1w)
{
    std::vector<double> c((size_t)nz * 12, 0.0);
    for (int k = 3; k <= nz - 2; ++k) {
        double delta = dz1w[k - 1], deltam1 = dz1w[k - 2], deltap1 = dz1w[k], deltap2 = dz1w[k + 1];
        double *p = c.data() + 12 * (k - 1);
        p[0] = delta / (deltam1 + delta + deltap1);
        p[1] = (2.0 * deltam1 + delta) / (deltap1 + delta);
        p[2] = (delta + 2.0 * deltap1) / (deltam1 + delta);
        p[3] = deltap1 / (delta + deltap1 + deltap2);
        p[4] = (2.0 * delta + deltap1) / (deltap2 + deltap1);
        p[5] = (deltap1 + 2.0 * deltap2) / (delta + deltap1);
        p[6] = delta / (delta + deltap1);
        p[7] = 1.0 / (deltam1 + delta + deltap1 + deltap2);
        p[8] = 2.0 * deltap1 * delta / (delta + deltap1) *
               ((deltam1 + delta) / (2.0 * delta + deltap1) - (deltap2 + deltap1) / (2.0 * deltap1 + delta));
        p[9] = delta * (deltam1 + delta) / (2.0 * delta + deltap1);
        p[10] = deltap1 * (deltap1 + deltap2) / (2.0 * deltap1 + delta);
    }
    return c;
}

}  // namespace mimadv
