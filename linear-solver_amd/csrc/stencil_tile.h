// stencil_tile.h -- the FD12 stencil sweep for grids too small to fill the
// chip with z-marching blocks.
//
// The march of stencil_body.h wants one deep column per CU: on a grid of a
// few million points it leaves most CUs idle and walks its planes one
// barrier at a time.  Here a block of WY wavefronts takes a BX x TY x LZ box
// and stages all its planes at once: every thread issues the loads of its PY
// columns of vectors (LZ + 2R planes, kept in registers for the
// z-neighbours) and of its share of the x/y halo vectors, parks the box
// planes with their halos in LDS, and after ONE barrier computes its
// PY*LZ*V points.  The price is (LZ + 2R)/LZ reads per point, from the caches
// at these sizes.
#pragma once

#include "stencil_point.h"

namespace aar {

template <typename T, int WY, int PY, int LZ> struct Tile {
    using L = Lane<T>;
    static constexpr int NT = 64 * WY;
    static constexpr int BX = tile_x<T>(LZ), LPR = BX / L::V, RPW = 64 / LPR;
    static constexpr int LW = BX + 2 * L::HXV * L::V;
    static constexpr int TY = WY * RPW * PY;
    static constexpr int LH = TY + 2 * R;
    static constexpr int NYC = 2 * R * LPR, NXC = TY * 2 * L::HXV;
    static constexpr int NHC = LZ * (NYC + NXC);                   // halo vectors of the box
    static constexpr int NH = (NHC + NT - 1) / NT;
    struct Lds {
        typename L::Vec tile[LZ * LH][LW / L::V];
        double red[2 * WY];
    };
};

template <typename T, int WY, int PY, int LZ, SMode MODE, bool VC, int XM>
__device__ __forceinline__ void stencil_box(const SArgs<T> &a, const int item, typename Tile<T, WY, PY, LZ>::Lds &S)
{
    using B = Tile<T, WY, PY, LZ>;
    using L = Lane<T>;
    using Vec = typename L::Vec;
    using Off = VOff<T, XM>;
    constexpr int V = L::V, LPR = B::LPR, HXV = L::HXV, BX = B::BX;
    constexpr int NT = B::NT, TY = B::TY, NHC = B::NHC, NH = B::NH;
    constexpr int NE = ModeInfo<MODE>::NE;
    constexpr int NACC = ModeInfo<MODE>::NACC;
    constexpr int NQ = LZ + 2 * R;                                 // planes of a column

    const int itx = item % a.ntx;
    const int rest = item / a.ntx;
    const int ity = rest % a.nty;
    const int izc = rest / a.nty;
    int x0, own;
    tile_x0<T, BX, XM>(itx, a.nx, x0, own);
    const int y0 = ity * TY, z0 = izc * LZ;
    const int tid = threadIdx.x, lane = tid & 63;
    const int xv = lane % LPR;
    const int r0 = ((tid >> 6) * B::RPW + lane / LPR) * PY;
    const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = a.nxy;

    const PointK<T> k(a);

    Off c_off[PY];
    bool c_ok[PY][V], s_ok[PY][V];                                 // norm terms; stores
#pragma unroll
    for (int p = 0; p < PY; p++) {
        c_off[p].set(x0 + xv * V, y0 + r0 + p, nx, ny);
#pragma unroll
        for (int v = 0; v < V; v++) {
            const int gx = x0 + xv * V + v;
            s_ok[p][v] = gx < nx && y0 + r0 + p < ny;
            c_ok[p][v] = s_ok[p][v] && gx >= own;
        }
    }
    // element offsets of the planes z0-R .. z0+LZ-1+R (wrapped; uniform)
    size_t zo[NQ];
    {
        int z = modp(z0 - R, nz);
#pragma unroll
        for (int s = 0; s < NQ; s++) {
            zo[s] = (size_t)z * nxy;
            z = z + 1 == nz ? 0 : z + 1;
        }
    }
    Vec q[PY][NQ];
#pragma unroll
    for (int s = 0; s < NQ; s++)
#pragma unroll
        for (int p = 0; p < PY; p++) q[p][s] = ld_vec<T, XM>(a.in0 + zo[s], c_off[p]);
    // halo vector c of the box: plane, then 2R rows of LPR and TY rows of
    // HXV left and HXV right
    Vec h[NH];
    int h_row[NH], h_col[NH];                                      // row over all planes of the LDS tile
#pragma unroll
    for (int j = 0; j < NH; j++) {
        const int c0 = tid + NT * j;
        const int cc = c0 < NHC ? c0 : 0;
        const int s = cc / (B::NYC + B::NXC), c = cc % (B::NYC + B::NXC);
        Off off;
        if (c < B::NYC) {
            const int r = c / LPR, w = c % LPR;
            off.set(x0 + w * V, r < R ? y0 - R + r : y0 + TY + (r - R), nx, ny);
            h_row[j] = s * B::LH + (r < R ? r : TY + r);
            h_col[j] = HXV + w;
        } else {
            const int r = (c - B::NYC) / (2 * HXV), w = (c - B::NYC) % (2 * HXV);
            off.set(w < HXV ? x0 - (HXV - w) * V : x0 + BX + (w - HXV) * V, y0 + r, nx, ny);
            h_row[j] = s * B::LH + R + r;
            h_col[j] = w < HXV ? w : LPR + w;
        }
        // the plane differs between lanes: part of the 32-bit offset
        const unsigned zs = (unsigned)modp(z0 + s, nz) * (unsigned)nxy;
#pragma unroll
        for (int v = 0; v < Off::NO; v++) off.o[v] += zs;
        h[j] = ld_vec<T, XM>(a.in0, off);
    }
    Vec en[PY][LZ], vv[PY][LZ];
    if constexpr (NE > 0) {
#pragma unroll
        for (int s = 0; s < LZ; s++)
#pragma unroll
            for (int p = 0; p < PY; p++) en[p][s] = ld_vec<T, XM>(a.bvec + zo[R + s], c_off[p]);
    }
    if constexpr (VC) {
#pragma unroll
        for (int s = 0; s < LZ; s++)
#pragma unroll
            for (int p = 0; p < PY; p++) vv[p][s] = ld_vec<T, XM>(a.vf + zo[R + s], c_off[p]);
    }

#pragma unroll
    for (int s = 0; s < LZ; s++)
#pragma unroll
        for (int p = 0; p < PY; p++) S.tile[s * B::LH + R + r0 + p][HXV + xv] = q[p][R + s];
#pragma unroll
    for (int j = 0; j < NH; j++)
        if (tid + NT * j < NHC) S.tile[h_row[j]][h_col[j]] = h[j];
    __syncthreads();

    double acc[NACC];
#pragma unroll
    for (int j = 0; j < NACC; j++) acc[j] = 0.0;
#pragma unroll
    for (int s = 0; s < LZ; s++) {
        if (z0 + s < nz) {                                         // uniform: planes past the grid
#pragma unroll
            for (int p = 0; p < PY; p++) {
                const int lr = s * B::LH + R + r0 + p;
                const Vec u = q[p][R + s];
                T xw[(2 * HXV + 1) * V];
#pragma unroll
                for (int w = 0; w < 2 * HXV + 1; w++) {
                    const Vec t = w == HXV ? u : S.tile[lr][xv + w];
#pragma unroll
                    for (int v = 0; v < V; v++) xw[w * V + v] = t[v];
                }
                // rows of this thread from its registers, the others from LDS
                auto yn = [&](int d) -> Vec {
                    const int pp = p + d;
                    if (pp >= 0 && pp < PY) return q[pp < 0 ? 0 : (pp < PY ? pp : PY - 1)][R + s];
                    return S.tile[lr + d][HXV + xv];
                };
                auto zn = [&](int d) -> Vec { return q[p][R + s + d]; };
                const Vec y = stencil_value<T, MODE, VC>(a, k, xw, vv[p][s], yn, zn);
                // PGR's two outputs wait a projection cycle: non-temporal
                // (128^3 103.2 -> 100.5 ms a solve; the other modes' output
                // is the next sweep's input, and they lose 0.3%)
                constexpr bool NT_OUT = MODE == SMode::PGR_STEP;
                auto put = [&](auto *base, const auto &o) {
                    st_vec<std::remove_pointer_t<decltype(base)>, NT_OUT, T, XM>(base + zo[R + s], c_off[p], o,
                                                                                  s_ok[p], true);
                };
                stencil_epilogue<T, MODE, VC, XM>(a, k, y, u, en[p][s], vv[p][s], c_ok[p], put, acc);
            }
        }
    }
    if (a.partials) block_reduce_to<NACC, NT>(acc, a.partials + (size_t)item * NACC, S.red);
}

// Boxes of one plane run on grids of about a block a CU or fewer: registers for
// two waves a SIMD, so that every load is under way at once (an AAR iteration at
// 24 x 24 x 28 15.25 -> 15.05 us; with registers for more waves the loads went out
// in groups).
template <typename T, int WY, int PY, int LZ, SMode MODE, bool VC, int XM>
__global__ __launch_bounds__(64 * WY) __attribute__((amdgpu_waves_per_eu(1, LZ == 1 ? 2 : 8)))
void stencil_tile_kernel(const SArgs<T> a)
{
    __shared__ typename Tile<T, WY, PY, LZ>::Lds S;
    if (a.ctrl && a.ctrl->done) return;
    stencil_box<T, WY, PY, LZ, MODE, VC, XM>(a, xcd_item(blockIdx.x, a.nitems), S);
}

}  // namespace aar
