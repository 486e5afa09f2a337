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
#include "fused_march.hpp"

namespace mimadv {

namespace {

using namespace faces;

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
// Bound by VALU issue: the FP32 'weno' kernel takes 196 vector instructions
// per cell, three quarters of them the upwind faces, at 99 % of the issue
// rate of the clock it runs at (3.6 ms per stage for 15 species at
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

    const int tiles = A.ntx * A.nty;
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
    const int nf = sizeof(T) == 8 ? A.n64_active : A.n32_active;
    march_item<SCHEME, TX, TY, T, KC>(
        A, chunk, t, f0, min(nf, f0 + fpi),
        [&](int f, const T *&q, const T *&q0, T *&out) {
            if constexpr (sizeof(T) == 8) {
                q = A.q64[f];
                q0 = A.q0_64[f];
                out = A.out64[f];
            } else {
                q = A.q32[f];
                q0 = A.q0_32[f];
                out = A.out32[f];
            }
        },
        tile_lds, face_lds, vel_lds);
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
