// stencil_body.h -- the z-marching FD12 stencil sweep shared by the
// single-operator and the batched kernels (see stencil.hip for the design
// notes).
#pragma once

#include "stencil_point.h"

namespace aar {

// LDS of one march block: the double-buffered plane tile with its x/y halos
// and the halo ring.  Shared by the forms of a kernel that holds two of them.
template <typename T, int WY, int PY, int W> struct March {
    using L = Lane<T>;
    static constexpr int NT = 64 * WY;                       // threads: WY wavefronts stacked in y
    static constexpr int LPR = W / L::V, RPW = 64 / LPR;     // lanes a row, rows a wavefront
    static constexpr int LW = W + 2 * L::HXV * L::V;         // row pitch of the plane tile
    static constexpr int TY = WY * RPW * PY;
    static constexpr int LH = TY + 2 * R;
    static constexpr int NHC = 2 * R * LPR + TY * 2 * L::HXV;      // halo vectors of a plane
    static constexpr int NH = (NHC + NT - 1) / NT;           // per thread
    static constexpr int HR = R + 1;                         // halo ring depth (planes)
    struct Lds {
        typename L::Vec tile[2][LH][LW / L::V];
        // Halo cells are fetched R planes ahead, in the same step as the
        // neighbouring blocks fetch those lines as their own queue planes, so
        // that they are served from L2; each thread parks its cells here until
        // their plane is computed (slots private to the thread: no barrier).
        typename L::Vec ring[HR][NHC];
        double red[8 * WY];
    };
};

// The stencil sweep of one work item (a W x TY column over a z-chunk) of
// the operator and fields in `a`; shared by the single-operator kernel
// below and the batched kernel of batch.hip.  WY wavefronts, PY rows per
// thread.  VC: the variable-coefficient operator a*Lap + c(x), with a
// pointwise field a.vf read in the epilogue.
template <typename T, int WY, int PY, SMode MODE, bool VC, int XM, int W = TX>
__device__ __forceinline__ void stencil_march(const SArgs<T> &a, const int item,
                                              typename March<T, WY, PY, W>::Lds &S)
{
    static_assert(!VC || MODE != SMode::RESID, "no variable-coefficient RESID sweep");
    using M = March<T, WY, PY, W>;
    using L = Lane<T>;
    using Vec = typename L::Vec;
    using Off = VOff<T, XM>;
    constexpr int V = L::V, LPR = M::LPR, HXV = L::HXV;
    constexpr int NT = M::NT, TY = M::TY, NHC = M::NHC, NH = M::NH, HR = M::HR;
    constexpr int NE = ModeInfo<MODE>::NE;
    constexpr int NACC = ModeInfo<MODE>::NACC;
    constexpr int QN = 2 * R + 1;

    const int itx = item % a.ntx;
    const int rest = item / a.ntx;
    const int ity = rest % a.nty;
    const int izc = rest / a.nty;
    int x0, own;
    tile_x0<T, W, XM>(itx, a.nx, x0, own);
    const int y0 = ity * TY;
    const int z0 = izc * a.lz;
    const int z1 = min(z0 + a.lz, a.nz);
    const int tid = threadIdx.x, lane = tid & 63;
    const int xv = lane % LPR;                                     // vector of the row
    const int r0 = ((tid >> 6) * M::RPW + lane / LPR) * PY;        // first row of this thread
    const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = a.nxy;

    Off c_off[PY];
    bool c_ok[PY][V];
#pragma unroll
    for (int p = 0; p < PY; p++) {
        c_off[p].set(x0 + xv * V, y0 + r0 + p, nx, ny);
#pragma unroll
        for (int v = 0; v < V; v++) c_ok[p][v] = (x0 + xv * V + v >= own) && (x0 + xv * V + v < nx) && (y0 + r0 + p < ny);
    }
    // halo vectors: 2R rows of LPR, then TY rows of HXV left and HXV right;
    // cells past the halo load a valid (unused) address so that every load is
    // unconditional; only their LDS accesses are predicated
    Off h_off[NH];
    int h_row[NH], h_col[NH];
    bool h_ok[NH];
#pragma unroll
    for (int k = 0; k < NH; k++) {
        const int c0 = tid + NT * k;
        h_ok[k] = c0 < NHC;
        const int c = h_ok[k] ? c0 : 0;
        if (c < 2 * R * LPR) {
            const int r = c / LPR, w = c % LPR;
            h_off[k].set(x0 + w * V, r < R ? y0 - R + r : y0 + TY + (r - R), nx, ny);
            h_row[k] = r < R ? r : TY + r;
            h_col[k] = HXV + w;
        } else {
            const int r = (c - 2 * R * LPR) / (2 * HXV), w = (c - 2 * R * LPR) % (2 * HXV);
            h_off[k].set(w < HXV ? x0 - (HXV - w) * V : x0 + W + (w - HXV) * V, y0 + r, nx, ny);
            h_row[k] = R + r;
            h_col[k] = w < HXV ? w : LPR + w;
        }
    }

    const PointK<T> k(a);

    Vec q[PY][QN];
    // prefetch register set: halo + epilogue inputs of one plane and the
    // queue plane R ahead of it.  The loads of plane z+1 are issued while
    // plane z is computed; two sets alternate (the plane loop is unrolled by
    // two) so that no pending load is copied between registers.  (Two planes
    // ahead measured the same at 512^3, FP64: 436 against 435 us.)
    struct Pre {
        Vec qn[PY];
        Vec h[NH];
        Vec en[PY];
        Vec vv[PY];                                   // VC: a.vf at the plane
    };
    Pre s0, s1;

    // prologue: queue planes z0-R .. z0+R-1, halo vectors of planes z0 ..
    // z0+R-1 into the ring
    {
        int z = modp(z0 - R, nz);
#pragma unroll
        for (int s = 0; s < 2 * R; s++) {
            const size_t zo = (size_t)z * nxy;
            z = z + 1 == nz ? 0 : z + 1;
#pragma unroll
            for (int p = 0; p < PY; p++) q[p][s] = ld_vec<T, XM>(a.in0 + zo, c_off[p]);
            if (s >= R) {
#pragma unroll
                for (int j = 0; j < NH; j++) {
                    const Vec f = ld_vec<T, XM>(a.in0 + zo, h_off[j]);
                    if (h_ok[j]) S.ring[s - R][tid + NT * j] = f;
                }
            }
        }
    }
    // queue plane and halo vectors of plane zp+R, epilogue inputs of plane zp
    // (indices wrap, so the prefetch past the last plane is a harmless
    // unused load)
    int zq = modp(z0 + R, nz), zc = z0;               // the next plane to prefetch
    auto prefetch = [&](Pre &st) {
        const size_t oq = (size_t)zq * nxy, oc = (size_t)zc * nxy;
        zq = zq + 1 == nz ? 0 : zq + 1;
        zc = zc + 1 == nz ? 0 : zc + 1;
#pragma unroll
        for (int p = 0; p < PY; p++) st.qn[p] = ld_vec<T, XM>(a.in0 + oq, c_off[p]);
#pragma unroll
        for (int j = 0; j < NH; j++) st.h[j] = ld_vec<T, XM>(a.in0 + oq, h_off[j]);
        if constexpr (NE > 0) {
#pragma unroll
            for (int p = 0; p < PY; p++) st.en[p] = ld_vec<T, XM>(a.bvec + oc, c_off[p]);
        }
        if constexpr (VC) {
#pragma unroll
            for (int p = 0; p < PY; p++) st.vv[p] = ld_vec<T, XM>(a.vf + oc, c_off[p]);
        }
    };

    double acc[NACC];
#pragma unroll
    for (int j = 0; j < NACC; j++) acc[j] = 0.0;

    int rs = 0;                                       // ring slot of the current plane
    auto plane = [&](const int z, Pre &cur, Pre &nxt) {
        auto &tile = S.tile[(z - z0) & 1];
        // queue top <- plane z+R; LDS <- plane z (centre + halo)
#pragma unroll
        for (int p = 0; p < PY; p++) {
            q[p][2 * R] = cur.qn[p];
            tile[R + r0 + p][HXV + xv] = q[p][R];
        }
        // halo of plane z from the ring; park the vectors of plane z+R
        const int ws = rs == 0 ? HR - 1 : rs - 1;     // (rs + R) mod HR
#pragma unroll
        for (int j = 0; j < NH; j++)
            if (h_ok[j]) tile[h_row[j]][h_col[j]] = S.ring[rs][tid + NT * j];
#pragma unroll
        for (int j = 0; j < NH; j++)
            if (h_ok[j]) S.ring[ws][tid + NT * j] = cur.h[j];
        rs = rs + 1 == HR ? 0 : rs + 1;
        prefetch(nxt);
        __syncthreads();

        const size_t zoff = (size_t)z * nxy;
#pragma unroll
        for (int p = 0; p < PY; p++) {
            // rows one after the other: the LDS loads of all rows in flight
            // at once take the FP64 sweeps past 256 VGPRs
            if (p > 0) __builtin_amdgcn_sched_barrier(0);
            const int lr = R + r0 + p;
            const Vec u = q[p][R];
            T xw[(2 * HXV + 1) * V];
#pragma unroll
            for (int w = 0; w < 2 * HXV + 1; w++) {
                const Vec t = w == HXV ? u : tile[lr][xv + w];
#pragma unroll
                for (int v = 0; v < V; v++) xw[w * V + v] = t[v];
            }
            // y-neighbours at row offset d: rows of this thread come from
            // its own registers, the others from the LDS tile (p and d are
            // compile-time constants after unrolling, so this folds)
            auto yn = [&](int d) -> Vec {
                const int pp = p + d;
                if (pp >= 0 && pp < PY) return q[pp < 0 ? 0 : (pp < PY ? pp : PY - 1)][R];
                return tile[lr + d][HXV + xv];
            };
            auto zn = [&](int d) -> Vec { return q[p][R + d]; };
            const Vec y = stencil_value<T, MODE, VC>(a, k, xw, cur.vv[p], yn, zn);
            // outputs are next read a whole sweep later (beyond the caches
            // at the sizes where the march runs): non-temporal stores
            auto put = [&](auto *base, const auto &o) {
                st_vec<std::remove_pointer_t<decltype(base)>, true, T, XM>(base + zoff, c_off[p], o, c_ok[p], false);
            };
            stencil_epilogue<T, MODE, VC, XM>(a, k, y, u, cur.en[p], cur.vv[p], c_ok[p], put, acc);
        }
        // shift the queue one plane
#pragma unroll
        for (int p = 0; p < PY; p++)
#pragma unroll
            for (int s = 0; s < 2 * R; s++) q[p][s] = q[p][s + 1];
    };

    // named sets (not an array) keep every set in registers
    int z = z0;
    prefetch(s0);
    // the prologue's loads complete here, so the loop's memory waits are
    // set by its own steady state rather than by the prologue's order
    __builtin_amdgcn_s_waitcnt(0);
    for (; z + 1 < z1; z += 2) {
        plane(z, s0, s1);
        plane(z + 1, s1, s0);
    }
    if (z < z1) plane(z, s0, s1);

    if (a.partials) block_reduce_to<NACC, NT>(acc, a.partials + (size_t)item * NACC, S.red);
}

// the batch: systems of any sides in one launch
template <typename T, int WY, int PY, SMode MODE, bool WIDE>
__device__ __forceinline__ void stencil_any(const SArgs<T> &a, const int item)
{
    __shared__ typename March<T, WY, PY, TX>::Lds S;
    if constexpr (WIDE) stencil_march<T, WY, PY, MODE, false, XWIDE>(a, item, S);
    else if (x_mode<T>(a.nx, a.ny, TX) == XPOINT) stencil_march<T, WY, PY, MODE, false, XPOINT>(a, item, S);
    else stencil_march<T, WY, PY, MODE, false, XSHIFT>(a, item, S);
}

template <typename T, int WY, int PY, SMode MODE, bool VC, int XM, int W>
__global__ __launch_bounds__(64 * WY) void stencil_kernel(const SArgs<T> a)
{
    __shared__ typename March<T, WY, PY, W>::Lds S;
    if (a.ctrl && a.ctrl->done) return;
    stencil_march<T, WY, PY, MODE, VC, XM, W>(a, xcd_item(blockIdx.x, a.nitems), S);
}

}  // namespace aar
