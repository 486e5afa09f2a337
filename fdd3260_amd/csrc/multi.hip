// multi.hip -- one launch advecting many independent periodic subdomains.
//
// A batch of unequal subdomains (each with its own grid, metrics, FP32
// velocity, dt, scheme and set of FP32 fields) is advanced by one
// launch per Shu-Osher stage.  The subdomains' work items (a
// tile of columns and a chunk of levels) are numbered consecutively; a
// workgroup finds its subdomain by a binary search of the first work id of
// every subdomain, reads that subdomain's argument block from a device
// table, and runs the column march of the single-grid batched kernel
// (fused_march.hpp), so the results are the same bits.
//
// The tile shape is chosen per subdomain (TX x TY with TX*TY = 256:
// 16x16, 32x8, 64x4) so that small or narrow subdomains waste fewer lanes;
// every scheme and shape is an instance of its own in the kernel, with
// constant LDS offsets.  (One march with the shape in registers took 94
// registers and 11.41 ms for three stages of 48 subdomains of 48 to 192 columns a
// side, the instances 69 and 10.34 ms.)  25 KB of LDS: six groups a CU.
// Bound by VALU issue, like the single-grid kernel.
#include <algorithm>
#include <type_traits>

#include "fused_march.hpp"

namespace mimadv {

namespace {

using namespace faces;

constexpr int NT = MULTI_NT;
constexpr int KC = MULTI_KC;  // levels of a work item (velocities staged in LDS)

// LDS of the largest shape
constexpr int TILE_MAX = Item<64, 4, 3>::LH * Item<64, 4, 3>::LW;
constexpr int FACE_MAX = Item<64, 4, 3>::NFACE;
constexpr int NV_MAX = Item<64, 4, 3>::NV;

__global__ __launch_bounds__(NT) void multi_kernel(const FusedArgs *__restrict__ table, int ndom)
{
    __shared__ float tile_lds[TILE_MAX];
    __shared__ float face_lds[FACE_MAX];
    __shared__ float vel_lds[KC * NV_MAX];
    const int wi = blockIdx.x;
    // subdomain of this work id: last d with work_begin <= wi
    int lo = 0, hi = ndom - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (table[mid].work_begin <= wi) lo = mid;
        else hi = mid - 1;
    }
    // a private copy of the argument block: its scalars stay in registers
    // instead of being reloaded after every store (the table is global
    // memory); the field pointers are read from the table once per field
    const FusedArgs A = table[lo];
    // fields f0 .. f1 - 1, level chunk and tile of the item
    const int tiles = A.ntx * A.nty, nchunk = (A.nz + A.kchunk - 1) / A.kchunk;
    int t = wi - A.work_begin;
    const int fg = t / (tiles * nchunk);
    t -= fg * tiles * nchunk;
    const int chunk = t / tiles;
    t -= chunk * tiles;
    const int f0 = fg * A.fpi, f1 = min(A.n32_active, f0 + A.fpi);
    const auto fields = [&](int f, const float *&q, const float *&q0, float *&out) {
        q = table[lo].q32[f];
        q0 = table[lo].q0_32[f];
        out = table[lo].out32[f];
    };
    const auto shape = [&](auto scheme) {
        constexpr int S = decltype(scheme)::value;
        if (A.tile_x == 32)
            march_item<S, 32, 8, float, KC>(A, chunk, t, f0, f1, fields, tile_lds, face_lds, vel_lds);
        else if (A.tile_x == 16)
            march_item<S, 16, 16, float, KC>(A, chunk, t, f0, f1, fields, tile_lds, face_lds, vel_lds);
        else
            march_item<S, 64, 4, float, KC>(A, chunk, t, f0, f1, fields, tile_lds, face_lds, vel_lds);
    };
    if (A.scheme == 0) shape(std::integral_constant<int, 0>{});
    else if (A.scheme == 3) shape(std::integral_constant<int, 3>{});
    else shape(std::integral_constant<int, 2>{});
}

}  // namespace

bool multi_tile_ok(int tile_x, int tile_y)
{
    return tile_x * tile_y == MULTI_NT && (tile_x == 16 || tile_x == 32 || tile_x == 64);
}

void multi_prepare(FusedArgs &A, int work_begin, int split)
{
    A.ntx = (A.nx - 5 + A.tile_x - 1) / A.tile_x;
    A.nty = (A.ny - 5 + A.tile_y - 1) / A.tile_y;
    A.kchunk = A.kchunk <= 0 ? KC : min(A.kchunk, KC);
    const int nf = std::max(1, A.n32_active);
    split = std::min(split, nf);
    A.fpi = (nf + split - 1) / split;
    A.nwork = A.ntx * A.nty * ((A.nz + A.kchunk - 1) / A.kchunk) * ((nf + A.fpi - 1) / A.fpi);
    A.work_begin = work_begin;
}

// Few subdomains leave the chip idle if every item marches all fields: the
// fields are then split so that the launch has eight groups per CU, as in the
// single-grid kernel (two subdomains of 48 to 60 columns a side, SSP-RK3 step
// 455 -> 177 us; from eight groups per CU on nothing is split).
int multi_number(std::vector<FusedArgs> &table)
{
    int work = 0;
    for (int split = 1;;) {
        work = 0;
        for (FusedArgs &A : table) {
            multi_prepare(A, work, split);
            work += A.nwork;
        }
        if (split > 1 || work == 0) return work;
        split = (8 * device_cus() + work - 1) / work;
        if (split <= 1) return work;
    }
}

hipError_t launch_multi(const FusedArgs *d_table, int ndom, int nwork, hipStream_t s)
{
    if (ndom <= 0 || nwork <= 0) return hipSuccess;
    // One group per work item, handed out by the hardware as CUs have room:
    // items differ in cost (schemes, field counts, ragged chunks), and a
    // resident grid of ncu * occupancy groups with a fixed share each ended
    // with most CUs idle (48 subdomains of 48 to 192 columns a side, three
    // SSP-RK3 stages: 13.18 -> 11.43 ms).
    hipLaunchKernelGGL(multi_kernel, dim3(nwork), dim3(NT), 0, s, d_table, ndom);
    return hipGetLastError();
}

}  // namespace mimadv
