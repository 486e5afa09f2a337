// fused_march.hpp -- a work item of the batched kernels: a tile of columns and
// a chunk of levels, marched by a workgroup for one field after the other.
// Shared by the single-grid (fused.hip) and multi-domain (multi.hip) kernels.
#pragma once
#include "fused.hpp"
#include "fused_faces.hpp"
#include "mimadv_internal.hpp"

namespace mimadv {
namespace faces {

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

// This thread's part of the halo of a work item's tile, the same for every
// field and level: offsets in a level plane (32 bits; threads past the end of
// the list load its last value) and in the LDS tile (-1 past the end).  The
// list holds the H columns west and east of every row, then the H rows south
// and north of every column; no face reads a corner.
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

// Work item (chunk, tile t) for fields f0 .. f1-1: fields(f, q, q0, out) gives
// a field's arrays; lt, lf and lv are the item's LDS (tile, faces, velocities
// of up to KC levels).
template <int SCHEME, int TX, int TY, class T, int KC, class Fields>
__device__ __forceinline__ void march_item(const FusedArgs &A, int chunk, int t, int f0, int f1, Fields fields, T *lt,
                                           T *lf, float *lv)
{
    constexpr int H = stencil_h<SCHEME>();
    using I = Item<TX, TY, H>;
    const int nx = A.nx, ny = A.ny, nz = A.nz;
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int i0 = 4 + (t % A.ntx) * TX;
    const int j0 = I::THREE_D ? 4 + (t / A.ntx) * TY : 1;
    const int k0 = 1 + chunk * A.kchunk;
    const int nk = min(A.kchunk, nz - k0 + 1);
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
                float *l = lv + kk * I::NV;
                l[tid] = vu[kk];
                if (I::THREE_D) l[I::SOUTH + tid] = vv[kk];
                if (rest) l[I::REST + tid] = vr[kk];
                l[I::NFACE + tid] = vw[kk];
            }
        __syncthreads();
    }
#pragma unroll 1
    for (int f = f0; f < f1; ++f) {
        const T *q, *q0;
        T *out;
        fields(f, q, q0, out);
        march_field<SCHEME, TX, TY, T>(A, q, q0, out, lt, lf, lv, k0, nk, i0, j0, tid, tx, ty, valid, col, halo);
    }
}

}  // namespace faces
}  // namespace mimadv
