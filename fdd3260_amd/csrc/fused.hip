// fused.hip -- batched, mixed-precision scalar advection on gfx950.
//
// One launch advects a batch of fields that share one velocity
// (u, v, w in FP32): up to MAX64 fields in FP64 (theta, water vapour: small
// increments on large values) and the rest in FP32.  A work item is a
// TX x TY tile of columns and a chunk of KC levels:
//
//   * the chunk's face velocities are staged in LDS once and serve every
//     field of the batch (fields are the outer loop, levels the inner one,
//     so register use does not grow with the field count);
//   * per field and level the tile plus a 2-cell halo goes through LDS (a
//     thread's own value from its column window, the halo requested a level
//     ahead), every thread forms the west and south face of its cell, one
//     wave the faces beyond the last column and row, and the z face k+1/2
//     of every column comes from a register window q(k-1..k+2) and is
//     carried to level k+1 as its bottom face;
//   * face fluxes of FP32 fields are FP32; the flux differences and the
//     divergence are accumulated in FP64 (exact differences of FP32 values,
//     a compensated sum) and the Shu-Osher stage update
//     q_new = c0*q0 + c1*(q + dt*div) is evaluated in FP64 and rounded once.
//
// Schemes: the reference WENO ('weno' of advq_weno.f90, including its
// limiter, the k = 3..nz-3 range of nonlinear vertical weights and the
// bottom/top closures), MUSCL (advq_muscl.f90) and the WENO5-JS extension
// (3-cell halo, in z where the upwind stencil fits the column) in an
// operation-reduced form: limiter_weno's rescale is applied to the
// weighted face value in a form that resolves its eps scale in FP32 (see
// weno_face), only the upwind side's weights are evaluated, and divisions
// are reciprocals.  It is checked against the FP64 oracle with tolerances,
// not bit for bit.  Vertical boundaries must be no-flux ('nnf'), the
// lateral ones periodic.
#include "fused.hpp"
#include "fused_faces.hpp"
#include "mimadv_internal.hpp"

namespace mimadv {

namespace {

using namespace faces;

// Geometry of one work item (a TX x TY column tile and a chunk of at most
// KC levels) shared by every field it advects.  A thread owns the cell (tx,
// ty), its west face and its south face; the faces beyond the tile's last
// column and row are `LO` left-over ones.
template <int TX, int TY, int H>
struct Item {
    static constexpr bool THREE_D = TY > 1;
    static constexpr int NT = TX * TY;
    static constexpr int LW = TX + 2 * H, LH = THREE_D ? TY + 2 * H : 1;  // tile + H-cell halo
    static constexpr int LO = TY + (THREE_D ? TX : 0);                   // east faces, then north faces
    static constexpr int NH = 2 * H * (TY + (THREE_D ? TX : 0));         // halo values (no corners)
    static constexpr int HS = (NH + NT - 1) / NT;                        // halo slots per thread
    static constexpr int NFACE = (THREE_D ? 2 * NT : NT) + LO;           // west, south, left-over
    static constexpr int SOUTH = NT, REST = THREE_D ? 2 * NT : NT;       // their offsets
    static constexpr int NV = NFACE + NT;                                // velocities per level: faces, then w
};

// Levels of a work item whose velocities are staged in LDS once and read by
// every field (the chunk length is capped at this).
constexpr int FUSED_KC = 8;

// The 256-thread tiles take shorter chunks: their LDS bounds how many groups
// share a CU, and more groups hide more than the velocity staging of a longer
// chunk saves.  FP32 six levels (23 KB, seven groups; WENO5 24 KB, six), FP64
// five (24 KB, six groups).  A step of 20 fields at 512x512x160: 6 and 8
// levels 15.54 ms, 6 and 5 15.44, 5 and 8 15.51, 4 and 8 15.65, 8 and 8 16.24;
// ten WENO5 species with two FP64 fields at 256x256x128: 8 and 8 1.08 ms, 6 and 5 1.02.
template <int SCHEME, int TX, int TY, class T>
constexpr int fused_kc()
{
    return TX * TY != 256 ? FUSED_KC : sizeof(T) == 8 ? 5 : 6;
}

// This thread's part of the halo of a work item's tile, the same for every
// field and level: offsets in a level plane (32 bits; threads past the end of the list
// load their own column) and in the LDS tile.  The list holds the H columns west and east of
// every row, then the H rows south and north of every column; no face reads a
// corner.
template <int TX, int TY, int H>
struct Halo {
    using I = Item<TX, TY, H>;
    int off[I::HS], pos[I::HS];
    __device__ __forceinline__ void init(int tid, int i0, int j0, const FusedArgs &A)
    {
#pragma unroll
        for (int s = 0; s < I::HS; ++s) {
            const int e = tid + s * I::NT, el = min(e, I::NH - 1);
            int r, c;
            if (el < 2 * H * TY) {
                r = el / (2 * H) + (I::THREE_D ? H : 0);
                c = el % (2 * H);
                c = c < H ? c : c + TX;
            } else {
                const int e2 = el - 2 * H * TY;
                r = e2 / TX;
                r = r < H ? r : r + TY;
                c = e2 % TX + H;
            }
            const int ii = wrap(i0 - H + c, A.nx, A.mx), jj = I::THREE_D ? wrap(j0 - H + r, A.ny, A.my) : 1;
            off[s] = (ii - 1) + A.nx * (jj - 1);
            pos[s] = e < I::NH ? r * I::LW + c : -1;
        }
    }
};

// One field marched up the item's levels.  Per level the tile goes to LDS (a
// thread's own value from its column window, the halo as requested one level
// ahead), every thread forms the west and south face of its cell and the top
// face of its column (register window q(k-H+1..k+H)), one wave the left-over
// faces; the faces of the eastern and northern neighbours come through LDS.
// Then the cell: FP64 flux divergence of the FP32/FP64 face values and the
// Shu-Osher stage update, rounded once to the field's precision, with the
// periodic ghost images.
template <int SCHEME, int TX, int TY, class T>
__device__ __forceinline__ void march_field(const FusedArgs &A, const T *__restrict__ q, const T *__restrict__ q0,
                                            T *__restrict__ out, T *lt, T *lf, const float *lv, int k0, int nk,
                                            int i0, int j0, int tid, int tx, int ty, bool valid, int col,
                                            const Halo<TX, TY, stencil_h<SCHEME>()> &halo)
{
    constexpr int H = stencil_h<SCHEME>();
    using I = Item<TX, TY, H>;
    const int nx = A.nx, ny = A.ny, nz = A.nz;
    const size_t plane = (size_t)nx * ny;
    auto lev = [&](int kk) { return (size_t)(min(max(kk, 1), nz) - 1) * plane; };
    // A chunk above the floor first evaluates its bottom face k0-1/2 in a
    // z-only pass of the level loop (kk = -1), so that every z face of the
    // column is evaluated by the same code whatever the chunking.
    const bool zdir = (A.dirmask & 4) != 0;
    const int kstart = (k0 > 1 && zdir) ? -1 : 0;
    const int ks = k0 + kstart;
    // byte offsets in a level plane: this thread's column, its halo slots
    uint32_t colb = (uint32_t)col * (uint32_t)sizeof(T);
    uint32_t hb[I::HS];
#pragma unroll
    for (int s = 0; s < I::HS; ++s) hb[s] = (uint32_t)halo.off[s] * (uint32_t)sizeof(T);
    // own position in the tile, and where the eastern and northern faces lie
    const int own = (I::THREE_D ? (ty + H) * I::LW : 0) + tx + H;
    const int fe = tx < TX - 1 ? tid + 1 : I::REST + ty;
    const int fn = ty < TY - 1 ? I::SOUTH + tid + TX : I::REST + TY + tx;
    // window q(ks-H+1..ks+H), levels outside 1..nz clamped
    T zw[2 * H];
#pragma unroll
    for (int m = 0; m < 2 * H; ++m) zw[m] = load_at(q + lev(ks - H + 1 + m), colb);
    const float wz0 = load_at(A.w + lev(ks + 1), (uint32_t)col * 4u);
    T fzb = T(0);
    T hv[I::HS];
    T q0v = T(0), zn = T(0);
    double d1v = 0.0;
    const bool need_q0 = A.epi != 0 && A.c0 != 0.0;
    // everything level k needs from memory, requested one level ahead; zn
    // = q(k+H) enters the window after level k-1
    auto fetch = [&](int k) {
        const size_t kb = lev(k);
        const T *qk = q + kb;
#pragma unroll
        for (int s = 0; s < I::HS; ++s) hv[s] = load_at(qk, hb[s]);
        if (need_q0) q0v = load_at(q0 + kb, colb);
        zn = load_at(q + lev(k + H), colb);
        d1v = table(A.dz1w)[k - 1];
    };
    fetch(k0);
    // waited for here: the waits in the loop then count what a level has in
    // flight itself, not the fewer requests of the way into it
#pragma unroll
    for (int s = 0; s < I::HS; ++s) settle(hv[s]);
    settle(q0v);
    settle(zn);
#pragma unroll 1
    for (int kk = kstart; kk < nk; ++kk) {
        const int k = k0 + kk;
        // opaque per level: otherwise every array's 64-bit address is hoisted
        // out of the loop into registers of its own
#pragma unroll
        for (int s = 0; s < I::HS; ++s) asm volatile("" : "+v"(hb[s]));
        asm volatile("" : "+v"(colb));
        // window q(k-H+1..k+H); this level's staged velocities
        const float *lvk = lv + (kk < 0 ? 0 : kk) * I::NV;
        const T fzt = zdir ? zface<SCHEME, T>(k, nz, zw, T(kk < 0 ? wz0 : lvk[I::NFACE + tid]), A) : T(0);
        if (kk >= 0) {
            lt[own] = zw[H - 1];
#pragma unroll
            for (int s = 0; s < I::HS; ++s)
                if (halo.pos[s] >= 0) lt[halo.pos[s]] = hv[s];
            const T q0c = q0v;
            const double dz1w_k = d1v;
            __syncthreads();
            fetch(k0 + min(kk + 1, nk - 1));
            // a face at a time, each from its own loads: values shared by two
            // faces would be fused into other multiply-adds in one than in the
            // other, and the bits would depend on the tile
            T sv[2 * H], fs = T(0);
#pragma unroll
            for (int m = 0; m < 2 * H; ++m) sv[m] = lt[own - H + m];
            T fw = hface<SCHEME, T>(sv, T(lvk[tid]), A, A.dx1);
            settle(fw);
            lf[tid] = fw;
            if constexpr (I::THREE_D) {
#pragma unroll
                for (int m = 0; m < 2 * H; ++m) sv[m] = lt[own + (m - H) * I::LW];
                fs = hface<SCHEME, T>(sv, T(lvk[I::SOUTH + tid]), A, A.dy1);
                settle(fs);
                lf[I::SOUTH + tid] = fs;
            }
            // the left-over faces, by another wave each level
            const int lo = (tid + 64 * kk) & (I::NT - 1);
            if (lo < I::LO) {
                const bool east = lo < TY;
                const int b = east ? (I::THREE_D ? (lo + H) * I::LW : 0) + TX : TY * I::LW + lo - TY + H;
                const int st = east ? 1 : I::LW;
#pragma unroll
                for (int m = 0; m < 2 * H; ++m) sv[m] = lt[b + m * st];
                lf[I::REST + lo] = hface<SCHEME, T>(sv, T(lvk[I::REST + lo]), A, east ? A.dx1 : A.dy1);
            }
            __syncthreads();
            if (valid) {
                // flux divergence in FP64: the differences of FP32 face
                // values are exact there, and the three terms are summed
                // with one rounding per term (a compensated FP32 sum)
                double div = 0.0;
                if (A.dirmask & 1) div += (double(lf[fe]) - double(fw)) * A.dx1;
                if (I::THREE_D && (A.dirmask & 2)) div += (double(lf[fn]) - double(fs)) * A.dy1;
                if (A.dirmask & 4) div += (double(fzt) - double(fzb)) * dz1w_k;
                const double a = -div;
                T *outk = out + (size_t)(k - 1) * plane;
                if (A.epi == 0) {
                    store_at(outk, colb, T(a));
                } else {
                    // Shu-Osher stage in FP64, rounded once
                    double qn;
                    if (A.c0 != 0.0) qn = A.c0 * double(q0c) + A.c1 * (double(zw[H - 1]) + A.dt * a);
                    else qn = A.c1 * (double(zw[H - 1]) + A.dt * a);
                    const T qv = T(qn);
                    store_at(outk, colb, qv);
                    if (A.fill) {
                        const int i = i0 + tx, j = j0 + ty;
                        int ix = 0, jy = 0;
                        if (i >= nx - 4) ix = i - A.mx;
                        else if (i <= 5) ix = i + A.mx;
                        if (I::THREE_D) {
                            if (j >= ny - 4) jy = j - A.my;
                            else if (j <= 5) jy = j + A.my;
                        }
                        const size_t kb = (size_t)(k - 1) * plane;
                        if (ix) out[kb + (size_t)(ix - 1) + (size_t)nx * (j - 1)] = qv;
                        if (jy) {
                            out[kb + (size_t)(i - 1) + (size_t)nx * (jy - 1)] = qv;
                            if (ix) out[kb + (size_t)(ix - 1) + (size_t)nx * (jy - 1)] = qv;
                        }
                    }
                }
            }
        }
        fzb = fzt;
#pragma unroll
        for (int m = 0; m < 2 * H - 1; ++m) zw[m] = zw[m + 1];
        zw[2 * H - 1] = zn;
    }
}

// LDS of a work item: a field's tile and faces of one level, the chunk's velocities.
template <int SCHEME, int TX, int TY, class T>
constexpr int fused_lds_bytes()
{
    using I = Item<TX, TY, stencil_h<SCHEME>()>;
    return (I::LH * I::LW + I::NFACE) * (int)sizeof(T) + fused_kc<SCHEME, TX, TY, T>() * I::NV * (int)sizeof(float);
}

// items: work items per group of fpi fields.  T: the precision of every field of the launch (FP64 and FP32 members of
// a batch go to two launches, so that the FP32 kernel keeps the register
// budget of FP32 arithmetic).
//
// Bound by VALU issue: the FP32 'weno' kernel takes about 190 vector
// instructions per cell, a third of them the upwind faces it cannot do
// without, at 85 % of the issue rate (3.6 ms per stage for 15 species at
// 512x512x160; a copy of its bytes takes 1.7 ms).  Faces by cell instead of a
// list of faces with their places in registers: constant LDS offsets, one
// plane offset for all of a thread's loads, 56 registers instead of 80 with
// spills; 16.0 -> 15.4 ms for a step of 20 fields with the chunks above, eight
// WENO5 species and two FP64 fields at 192x160x96 420 -> 360 us.
template <int SCHEME, int TX, int TY, class T>
__global__ __launch_bounds__(TX *TY) void fused_kernel(FusedArgs A, int items, int fpi)
{
    constexpr int H = stencil_h<SCHEME>();
    using I = Item<TX, TY, H>;
    __shared__ T tile_lds[I::LH * I::LW];
    __shared__ T face_lds[I::NFACE];
    constexpr int KC = fused_kc<SCHEME, TX, TY, T>();
    __shared__ float vel_lds[KC * I::NV];

    const int nx = A.nx, ny = A.ny, nz = A.nz;
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int tiles = A.ntx * A.nty;
    const int kc = A.kchunk;

    // fields f0 .. f0 + fpi - 1 of the batch
    const int fg = blockIdx.x / items, wi = blockIdx.x - fg * items;
    const int f0 = fg * fpi;
    // XCD-aware order: consecutive work ids go round-robin over the 8
    // XCDs; every XCD gets a contiguous range of tiles so that tile
    // halos and velocity rows stay in one L2.
    const int chunk = wi / tiles;
    int t = wi - chunk * tiles;
    if (A.xcd_remap) {
        const int per = tiles / 8;
        t = (t % 8) * per + t / 8;
    }
    const int i0 = 4 + (t % A.ntx) * TX;
    const int j0 = I::THREE_D ? 4 + (t / A.ntx) * TY : 1;
    const int k0 = 1 + chunk * kc;
    const int nk = min(kc, nz - k0 + 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool valid = i <= nx - 2 && (!I::THREE_D || j <= ny - 2);
    const int il = wrap(i, nx, A.mx), jl = I::THREE_D ? wrap(j, ny, A.my) : 1;
    const int col = (il - 1) + nx * (jl - 1);
    Halo<TX, TY, H> halo;
    halo.init(tid, i0, j0, A);
    // The chunk's face velocities and column w(k+1), read once for every
    // field: a thread's own west face, south face and column share one
    // plane offset, the left-over faces go to the first threads.  All the
    // chunk's loads are in flight together before they go to LDS.
    {
        const size_t plane = (size_t)nx * ny;
        const bool rest = tid < I::LO, east = tid < TY;
        const int ri = wrap(east ? i0 + TX : i0 + tid - TY, nx, A.mx);
        const int rj = I::THREE_D ? wrap(east ? j0 + tid : j0 + TY, ny, A.my) : 1;
        const int rcol = (ri - 1) + nx * (rj - 1);
        const float *rp = east ? A.u : A.v;
        float vu[KC], vv[KC], vr[KC], vw[KC];
#pragma unroll
        for (int kk = 0; kk < KC; ++kk) {
            const int k = k0 + kk;
            vu[kk] = vv[kk] = vr[kk] = vw[kk] = 0.0f;
            if (kk < nk) {
                const size_t kb = (size_t)(k - 1) * plane;
                vu[kk] = A.u[kb + col];
                if (I::THREE_D) vv[kk] = A.v[kb + col];
                if (rest) vr[kk] = rp[kb + rcol];
                if (k < nz) vw[kk] = A.w[kb + plane + col];  // w(k+1) at level k
            }
        }
#pragma unroll
        for (int kk = 0; kk < KC; ++kk)
            if (kk < nk) {
                float *l = vel_lds + kk * I::NV;
                l[tid] = vu[kk];
                if (I::THREE_D) l[I::SOUTH + tid] = vv[kk];
                if (rest) l[I::REST + tid] = vr[kk];
                l[I::NFACE + tid] = vw[kk];
            }
        __syncthreads();
    }
    if constexpr (sizeof(T) == 8) {
#pragma unroll 1
        for (int f = f0; f < min(A.n64_active, f0 + fpi); ++f)
            march_field<SCHEME, TX, TY, T>(A, A.q64[f], A.q0_64[f], A.out64[f], tile_lds, face_lds, vel_lds, k0, nk,
                                           i0, j0, tid, tx, ty, valid, col, halo);
    } else {
#pragma unroll 1
        for (int f = f0; f < min(A.n32_active, f0 + fpi); ++f)
            march_field<SCHEME, TX, TY, T>(A, A.q32[f], A.q0_32[f], A.out32[f], tile_lds, face_lds, vel_lds, k0, nk,
                                           i0, j0, tid, tx, ty, valid, col, halo);
    }
}

template <int SCHEME, int TX, int TY, class T>
hipError_t launch_tiles(const FusedArgs &a0, hipStream_t s, int blocks_per_cu)
{
    FusedArgs A = a0;
    A.ntx = (A.nx - 5 + TX - 1) / TX;
    A.nty = TY > 1 ? (A.ny - 5 + TY - 1) / TY : 1;
    const int tiles = A.ntx * A.nty;
    A.xcd_remap = (tiles % 8 == 0) ? 1 : 0;
    constexpr int KC = fused_kc<SCHEME, TX, TY, T>();
    // A grid whose items leave the chip idle splits the batch: each item then
    // marches fpi of the fields, so that FP32 launches have at least eight
    // 256-thread groups per CU (what makes a few ragged rounds cheap) and
    // FP64 ones the four that fit.  If one field per item does not give four
    // groups per CU, the chunks are shortened to reach them (unless the caller
    // set their length).  Every item stages the velocities of its chunk
    // again, so larger grids keep all fields in one item (256x256x128:
    // 1063 us, split further 1077).
    // Tendencies of 20 fields, all fields per item -> this rule: 24x24x16
    // 209 -> 86 us, 48x48x48 281 -> 171 us, 96x96x48 288 -> 207 us,
    // 192x160x96 536 -> 483 us.
    const int nf = sizeof(T) == 8 ? A.n64_active : A.n32_active;
    const long cus = (long)device_cus() * 256 / (TX * TY);
    const int kmax = A.kchunk <= 0 ? KC : min(A.kchunk, KC);
    const auto chunks = [&](int kc) { return (A.nz + kc - 1) / kc; };
    const long whole = (long)tiles * chunks(kmax), wide = (sizeof(T) == 8 ? 4 : 8) * cus;
    const int split = (int)max(1L, min((long)nf, (wide + whole - 1) / whole));
    const int fpi = (nf + split - 1) / split;
    const int groups = (nf + fpi - 1) / fpi;
    if (A.kchunk <= 0) {
        const int nchunk = (int)max((long)chunks(kmax), min((long)A.nz, 4 * cus / ((long)tiles * groups)));
        A.kchunk = (A.nz + nchunk - 1) / nchunk;
    } else A.kchunk = kmax;
    const int items = tiles * chunks(A.kchunk);
    A.nwork = items * groups;
    // One group per work item: the hardware hands the next item to the CU
    // that has room first.  A resident grid of ncu * occupancy groups, each
    // taking every gridDim-th item, leaves most CUs idle behind the longest
    // share: a step of 20 fields at 512x512x160 (three stages, momenta
    // included) took 18.55 ms that way and 16.02 ms this way.  A caller's
    // limit of groups per CU is kept by asking for that share of the LDS.
    int dyn = 0;
    if (blocks_per_cu > 0) {
        int dev = 0, most = 0, lds = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
            hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) == hipSuccess)
            dyn = max(0, min(most, lds / blocks_per_cu) - fused_lds_bytes<SCHEME, TX, TY, T>());
    }
    hipLaunchKernelGGL((fused_kernel<SCHEME, TX, TY, T>), dim3(A.nwork), dim3(TX * TY), dyn, s, A, items, fpi);
    return hipGetLastError();
}

template <int SCHEME, class T>
hipError_t launch_prec(const FusedArgs &A, hipStream_t s, int bpc)
{
    if (!A.three_d) return launch_tiles<SCHEME, 64, 1, T>(A, s, bpc);
    // default 32x8: the fewest x/y faces per cell of the 256-thread tiles
    // (552 for 256 cells against 580 for 64x4) and the smallest halo tile
    if (A.tile_x == 32 || (A.tile_x == 0 && A.tile_y == 0)) return launch_tiles<SCHEME, 32, 8, T>(A, s, bpc);
    if (A.tile_x == 16) return launch_tiles<SCHEME, 16, 16, T>(A, s, bpc);
    const int ty = A.tile_y > 0 ? A.tile_y : 4;
    switch (ty) {
    case 2: return launch_tiles<SCHEME, 64, 2, T>(A, s, bpc);
    case 4: return launch_tiles<SCHEME, 64, 4, T>(A, s, bpc);
    default: return launch_tiles<SCHEME, 64, 8, T>(A, s, bpc);
    }
}

template <int SCHEME>
hipError_t launch_scheme(const FusedArgs &A, hipStream_t s, int bpc)
{
    hipError_t e = hipSuccess;
    if (A.n64_active > 0) e = launch_prec<SCHEME, double>(A, s, bpc);
    if (e == hipSuccess && A.n32_active > 0) e = launch_prec<SCHEME, float>(A, s, bpc);
    return e;
}

}  // namespace

int fused_padded_count(int n32)
{
    return (n32 >= 0 && n32 <= FUSED_MAX32) ? n32 : -1;
}

hipError_t launch_fused(int scheme, int n64, int n32, const FusedArgs &A, hipStream_t s, int blocks_per_cu)
{
    if (n64 < 0 || n64 > FUSED_MAX64 || n32 < 0 || n32 > FUSED_MAX32) return hipErrorInvalidValue;
    if (scheme == 0) return launch_scheme<0>(A, s, blocks_per_cu);
    if (scheme == 2) return launch_scheme<2>(A, s, blocks_per_cu);
    if (scheme == 3) return launch_scheme<3>(A, s, blocks_per_cu);
    return hipErrorInvalidValue;
}

}  // namespace mimadv
