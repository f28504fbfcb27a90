// update.hip -- the pointwise steps of the solvers (Anderson and projection
// updates, CG), FP64 dots and the reductions' finishing kernel.
#include <algorithm>
#include <type_traits>

#include "history.h"

namespace aar {

// ---------------------------------------------------------------------------
// Anderson update (AAR.c:225-231 then AAR.c:116-117):
//   x_new = (x_k + beta f_k) - sum_k (DX_k + beta DF_k) s_col(k)
// The m-term sum runs in age order (the reference sums in column order;
// the two differ by summation order only).
// ---------------------------------------------------------------------------
template <typename T, int MM>
__global__ __launch_bounds__(BLOCK) void aar_update_kernel(const UpdArgs<T> a)
{
    constexpr int NS = MM + 1;
    if (a.ctrl->done) return;
    const int nv = a.nvalid, dir = a.direct;
    const T *px[NS], *pf[NS];
    bool use[NS];
    double sv[MM];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        use[k] = dir ? (k < nv) : (k <= nv);
        const size_t off = (size_t)(use[k] ? a.slot[k] : 0) * a.ld;
        px[k] = a.X + off;
        pf[k] = a.F + off;
    }
#pragma unroll
    for (int k = 0; k < MM; k++) sv[k] = k < nv ? a.ctrl->s[ref_col(a.it, k, a.m, dir)] : 0.0;
    const T *xk = dir ? a.X + (size_t)a.xslot * a.ld : px[0];
    const T *fk = dir ? a.F + (size_t)a.fslot * a.ld : pf[0];
    T *xo = const_cast<T *>(a.X) + (size_t)a.oslot * a.ld;
    const T beta = (T)a.beta;

    auto point = [&](T xb, T fb, const T (&vx)[NS], const T (&vf)[NS]) -> T {
        double am = 0.0;
#pragma unroll
        for (int k = 0; k < MM; k++) {
            if (k < nv) {
                const T dx = dir ? vx[k] : vx[k] - vx[k + 1];
                const T df = dir ? vf[k] : vf[k] - vf[k + 1];
                am = am + (double)(dx + beta * df) * sv[k];
            }
        }
        const T x0 = xb + beta * fb;
        return (T)((double)x0 - am);
    };

    const long n = a.n;
    const long stride = (long)gridDim.x * BLOCK;
    if ((n & 1) == 0) {
        using V2 = typename Vec2<T>::type;
        const long np = n >> 1;
        for (long ip = chunk_first(); ip < np; ip = chunk_next(ip)) {
            const long i = 2 * ip;
            T vx0[NS], vx1[NS], vf0[NS], vf1[NS];
#pragma unroll
            for (int k = 0; k < NS; k++) {
                vx0[k] = vx1[k] = vf0[k] = vf1[k] = (T)0;
                if (use[k]) {
                    const V2 u = *reinterpret_cast<const V2 *>(px[k] + i);
                    const V2 w = *reinterpret_cast<const V2 *>(pf[k] + i);
                    vx0[k] = u.x;
                    vx1[k] = u.y;
                    vf0[k] = w.x;
                    vf1[k] = w.y;
                }
            }
            V2 xb, fb;
            if (dir) {
                xb = *reinterpret_cast<const V2 *>(xk + i);
                fb = *reinterpret_cast<const V2 *>(fk + i);
            } else {
                xb.x = vx0[0];
                xb.y = vx1[0];
                fb.x = vf0[0];
                fb.y = vf1[0];
            }
            V2 o;
            o.x = point(xb.x, fb.x, vx0, vf0);
            o.y = point(xb.y, fb.y, vx1, vf1);
            *reinterpret_cast<V2 *>(xo + i) = o;
        }
    } else {
        for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) {
            T vx[NS], vf[NS];
#pragma unroll
            for (int k = 0; k < NS; k++) {
                vx[k] = use[k] ? px[k][i] : (T)0;
                vf[k] = use[k] ? pf[k][i] : (T)0;
            }
            xo[i] = point(xk[i], fk[i], vx, vf);
        }
    }
}

template <typename T>
hipError_t launch_aar_update(const UpdArgs<T> &a, hipStream_t st)
{
    if (a.m < 1 || a.m > MAXM || a.nvalid < 0 || a.nvalid > a.m) return hipErrorInvalidValue;
    long nb = (a.n / 2 + BLOCK - 1) / BLOCK;
    nb = nb < 1 ? 1 : (nb > 4096 ? 4096 : nb);
    if (a.m <= MAXM_FAST) hipLaunchKernelGGL((aar_update_kernel<T, MAXM_FAST>), dim3((unsigned)nb), dim3(BLOCK), 0, st, a);
    else if (a.m <= MAXM_MID) hipLaunchKernelGGL((aar_update_kernel<T, MAXM_MID>), dim3((unsigned)nb), dim3(BLOCK), 0, st, a);
    else hipLaunchKernelGGL((aar_update_kernel<T, MAXM>), dim3((unsigned)nb), dim3(BLOCK), 0, st, a);
    return hipGetLastError();
}
template hipError_t launch_aar_update<double>(const UpdArgs<double> &, hipStream_t);
template hipError_t launch_aar_update<float>(const UpdArgs<float> &, hipStream_t);

// ---------------------------------------------------------------------------
// Anderson step of the residual-recurrence AAR (AAR.c:109-117 with the
// iterates held as anchor + omega * g increments; see AncArgs).  The term
// coefficients are computed by every thread from uniform data (kernel
// arguments, ctrl->s) with static indices only, so they stay in registers
// without spills; NGM/NCM bound the term counts at compile time.
// ---------------------------------------------------------------------------
// Walks.  The arithmetic of each point is the same in every walk.
// * ONE (FP64 history, at most 8 residual terms and one correction): one
//   pair per thread and one block per NT pairs, x read and written
//   non-temporally (it is next read a whole cycle later); at 512^3 with
//   m = 7, p = 6 this took the update from 2.46 to 2.17 ms.
// * QUAD (FP32 history, FP64 x, the same term counts; the host checked
//   n % 4 == 0 and a 16-byte aligned x): four points per thread, 16-byte
//   history loads, one block per NT quads, every stream non-temporal
//   (1.35 -> 1.29 ms).  One pair per thread there halves the bytes a block
//   keeps in flight: 2.40 ms.
// * Otherwise (the wider forms, and FP32 history off those conditions):
//   chunks of CHUNK_V pairs, block b taking chunks b, b + grid, ..., over at
//   most 4096 blocks.  At 100-256 VGPRs one pair per thread measured 7.6
//   against 3.6 ms (m = 13, p = 11).
// * Odd n, or x off a pair: a grid stride of single points.
template <typename Tx, typename Tg, int NGM, int NCM, int NT, bool ONE, bool QUAD = false>
__global__ __launch_bounds__(NT) void anchor_update_kernel(const AncArgs<Tx, Tg> a)
{
    if (a.ctrl && a.ctrl->done) return;
    const int ng = a.ng, nc = a.nc;
    double cg[NGM], cc[NCM > 0 ? NCM : 1];
#pragma unroll
    for (int i = 0; i < NGM; i++) cg[i] = (a.with_beta && i == ng - 1) ? a.beta : 0.0;
#pragma unroll
    for (int c = 0; c < (NCM > 0 ? NCM : 1); c++) cc[c] = 0.0;
    for (int t = 0; t < a.ncol; t++) {
        const double gam = a.ctrl->s[a.col_ref[t]];
        const int j = a.col_j[t], cj = a.col_c[t];
#pragma unroll
        for (int i = 0; i < NGM; i++) {
            // dg_t = g_j - g_{j-1}; dx_t = omega g_{j-1} (Richardson step)
            if (i == j) cg[i] -= a.beta * gam;
            if (i == j - 1) cg[i] += (cj < 0) ? (a.beta - a.omega) * gam : a.beta * gam;
        }
#pragma unroll
        for (int c = 0; c < NCM; c++)
            if (c == cj) cc[c] -= gam;       // dx_t = an earlier Anderson correction
    }
    const int xlo = a.xlo, xhi = a.xhi;
    const double om = a.omega;
    Tg *co = (a.cout >= 0) ? a.C + (size_t)a.cout * a.ld : nullptr;

    const long n = a.n;
    if constexpr (QUAD) {
        static_assert(sizeof(Tg) == 4 && sizeof(Tx) == 8, "four-point form: FP32 history, FP64 x");
        typedef float F4 __attribute__((ext_vector_type(4)));
        typedef double D2 __attribute__((ext_vector_type(2)));
        const long iq = (long)blockIdx.x * NT + threadIdx.x;
        if (iq >= (n >> 2)) return;
        const long e = 4 * iq;
        F4 v[NGM];
#pragma unroll
        for (int i = 0; i < NGM; i++)
            if (i < ng) v[i] = __builtin_nontemporal_load(reinterpret_cast<const F4 *>(a.G + (size_t)a.gslot[i] * a.ld + e));
        F4 w[NCM > 0 ? NCM : 1];
#pragma unroll
        for (int c = 0; c < NCM; c++)
            if (c < nc) w[c] = __builtin_nontemporal_load(reinterpret_cast<const F4 *>(a.C + (size_t)a.cslot[c] * a.ld + e));
        const D2 x01 = __builtin_nontemporal_load(reinterpret_cast<const D2 *>(a.x + e));
        const D2 x23 = __builtin_nontemporal_load(reinterpret_cast<const D2 *>(a.x + e + 2));
        double sx[4] = {0.0, 0.0, 0.0, 0.0}, sc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < NGM; i++)
            if (i < ng) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const double g = (double)v[i][q];
                    if (i >= xlo && i < xhi) sx[q] += g;
                    sc[q] += cg[i] * g;
                }
            }
#pragma unroll
        for (int c = 0; c < NCM; c++)
            if (c < nc) {
#pragma unroll
                for (int q = 0; q < 4; q++) sc[q] += cc[c] * (double)w[c][q];
            }
        D2 o01, o23;
        o01.x = x01.x + (om * sx[0] + sc[0]);
        o01.y = x01.y + (om * sx[1] + sc[1]);
        o23.x = x23.x + (om * sx[2] + sc[2]);
        o23.y = x23.y + (om * sx[3] + sc[3]);
        __builtin_nontemporal_store(o01, reinterpret_cast<D2 *>(a.x + e));
        __builtin_nontemporal_store(o23, reinterpret_cast<D2 *>(a.x + e + 2));
        if (co) {
            F4 c4;
            c4.x = (float)sc[0];
            c4.y = (float)sc[1];
            c4.z = (float)sc[2];
            c4.w = (float)sc[3];
            __builtin_nontemporal_store(c4, reinterpret_cast<F4 *>(co + e));
        }
        return;
    }
    const long stride = (long)gridDim.x * NT;
    // pairs when n is even and x is aligned to a pair (ring slots always are)
    if ((n & 1) == 0 && ((uintptr_t)a.x % (2 * sizeof(Tx))) == 0) {
        using VX = typename Vec2<Tx>::type;
        using VG = typename Vec2<Tg>::type;
        const long np = n >> 1;
        for (long ip = ONE ? (long)blockIdx.x * NT + threadIdx.x : chunk_first(); ip < np;
             ip = ONE ? np : chunk_next(ip)) {
            const long e = 2 * ip;
            double sx0 = 0.0, sx1 = 0.0, sc0 = 0.0, sc1 = 0.0;
            VG v[NGM];
#pragma unroll
            for (int i = 0; i < NGM; i++)
                if (i < ng) v[i] = ld_nt2<VG>(a.G + (size_t)a.gslot[i] * a.ld + e);
            VG w[NCM > 0 ? NCM : 1];
#pragma unroll
            for (int c = 0; c < NCM; c++)
                if (c < nc) w[c] = ld_nt2<VG>(a.C + (size_t)a.cslot[c] * a.ld + e);
            const VX xv = ONE ? ld_nt2<VX>(a.x + e) : *reinterpret_cast<const VX *>(a.x + e);
#pragma unroll
            for (int i = 0; i < NGM; i++)
                if (i < ng) {
                    const double g0 = (double)v[i].x, g1 = (double)v[i].y;
                    if (i >= xlo && i < xhi) {
                        sx0 += g0;
                        sx1 += g1;
                    }
                    sc0 += cg[i] * g0;
                    sc1 += cg[i] * g1;
                }
#pragma unroll
            for (int c = 0; c < NCM; c++)
                if (c < nc) {
                    sc0 += cc[c] * (double)w[c].x;
                    sc1 += cc[c] * (double)w[c].y;
                }
            VX xo;
            xo.x = (Tx)((double)xv.x + (om * sx0 + sc0));
            xo.y = (Tx)((double)xv.y + (om * sx1 + sc1));
            if (ONE) st_nt2(a.x + e, xo);
            else *reinterpret_cast<VX *>(a.x + e) = xo;
            if (co) {
                VG c2;
                c2.x = (Tg)sc0;
                c2.y = (Tg)sc1;
                st_nt2(co + e, c2);
            }
        }
    } else {
        for (long e = (long)blockIdx.x * NT + threadIdx.x; e < n; e += stride) {
            double sx = 0.0, sc = 0.0;
#pragma unroll
            for (int i = 0; i < NGM; i++)
                if (i < ng) {
                    const double g = (double)a.G[(size_t)a.gslot[i] * a.ld + e];
                    if (i >= xlo && i < xhi) sx += g;
                    sc += cg[i] * g;
                }
#pragma unroll
            for (int c = 0; c < NCM; c++)
                if (c < nc) sc += cc[c] * (double)a.C[(size_t)a.cslot[c] * a.ld + e];
            a.x[e] = (Tx)((double)a.x[e] + (om * sx + sc));
            if (co) co[e] = (Tg)sc;
        }
    }
}

template <typename Tx, typename Tg>
hipError_t launch_anchor_update(const AncArgs<Tx, Tg> &a, hipStream_t st)
{
    if (a.ng < 1 || a.ng > NGMAX || a.nc < 0 || a.nc > NCMAX || a.ncol < 0 || a.ncol > MAXM)
        return hipErrorInvalidValue;
    if (a.xlo < 0 || a.xhi > a.ng || !a.G || !a.x) return hipErrorInvalidValue;
    if ((a.nc > 0 || a.cout >= 0) && !a.C) return hipErrorInvalidValue;
    if (a.ncol > 0 && !a.ctrl) return hipErrorInvalidValue;
    for (int t = 0; t < a.ncol; t++)
        if (a.col_j[t] < 1 || a.col_j[t] >= a.ng || a.col_c[t] >= a.nc || a.col_ref[t] < 0 ||
            a.col_ref[t] >= MAXM)
            return hipErrorInvalidValue;
    // FP64 history: one block per 1024 pairs where the terms are at most 8
    // residuals and one correction (m = 7, p = 6 among them).  FP32 history with FP64
    // x: four points per thread in that common form when n % 4 == 0 and x
    // is 16-byte aligned; otherwise a chunk walk over at most 4096 blocks.
    // The scalar fallback (odd n, x off a pair) walks a grid stride over
    // the same grid.
    constexpr bool ONE = sizeof(Tg) == 8;
    const long np = (a.n + 1) / 2;
    auto blocks = [np](long nt) {
        if (!ONE) {
            const long nb = (np + CHUNK_V - 1) / CHUNK_V;
            return (unsigned)(nb < 1 ? 1 : (nb > 4096 ? 4096 : nb));
        }
        return (unsigned)((np + nt - 1) / nt);
    };
    if (np > 0x7fffffffL * 256L) return hipErrorInvalidValue;
    constexpr int NT8 = ONE ? 1024 : BLOCK;
    if constexpr (sizeof(Tg) == 4 && sizeof(Tx) == 8) {
        // FP32 history, FP64 x: four points per thread where n and x allow
        // (ring slots are 256-byte aligned)
        if (a.ng <= 8 && a.nc <= 1 && a.n % 4 == 0 && (uintptr_t)a.x % 16 == 0) {
            const long nq = a.n / 4;
            hipLaunchKernelGGL((anchor_update_kernel<Tx, Tg, 8, 1, 1024, false, true>),
                               dim3((unsigned)((nq + 1023) / 1024)), dim3(1024), 0, st, a);
            return hipGetLastError();
        }
    }
    // the wider forms keep the chunk walk: at 100-256 VGPRs (2-3 waves per
    // SIMD) one pair per thread keeps too few bytes in flight (m = 13,
    // p = 11 at 512^3: 7.6 ms against 2.0 ms for the walk)
    const long nwalk = std::max(1L, std::min(4096L, (np + CHUNK_V - 1) / CHUNK_V));
    if (a.ng <= 8 && a.nc <= 1)
        hipLaunchKernelGGL((anchor_update_kernel<Tx, Tg, 8, 1, NT8, ONE>), dim3(blocks(NT8)), dim3(NT8), 0, st, a);
    else if (a.ng <= MAXM_FAST + 2 && a.nc <= MAXM_FAST + 1)
        hipLaunchKernelGGL((anchor_update_kernel<Tx, Tg, MAXM_FAST + 2, MAXM_FAST + 1, BLOCK, false>),
                           dim3((unsigned)nwalk), dim3(BLOCK), 0, st, a);
    else if (a.ng <= MAXM_MID + 2 && a.nc <= MAXM_MID + 1)
        hipLaunchKernelGGL((anchor_update_kernel<Tx, Tg, MAXM_MID + 2, MAXM_MID + 1, BLOCK, false>),
                           dim3((unsigned)nwalk), dim3(BLOCK), 0, st, a);
    else
        hipLaunchKernelGGL((anchor_update_kernel<Tx, Tg, NGMAX, NCMAX, BLOCK, false>), dim3((unsigned)nwalk),
                           dim3(BLOCK), 0, st, a);
    return hipGetLastError();
}
template hipError_t launch_anchor_update<double, double>(const AncArgs<double, double> &, hipStream_t);
template hipError_t launch_anchor_update<double, float>(const AncArgs<double, float> &, hipStream_t);
template hipError_t launch_anchor_update<float, float>(const AncArgs<float, float> &, hipStream_t);

// ---------------------------------------------------------------------------
// PGR / PL2R projection update (PGR.c:117-133): x += sum DX s; Ax += sum DF s
// in place at the age-0 slot; ||b - Ax||^2 for the convergence check; and the
// Richardson step of the next iteration, x + omega (b - Ax)/diag, into the
// slot `next` (one more vector written here; the sweep that would form it at
// every halo point reads two vectors less).
// Every stream is read and written non-temporally (each is next touched a
// whole sweep later).  ONE (m <= 8): one pair per thread, one block and one
// partial per NT pairs; at 512^3 with m = 7 this measured 3.71 ms against
// 4.11 ms for the chunk walk over 2048 blocks with plain accesses.  Deeper
// histories keep the chunk walk (BLOCK threads, many more registers).
// ---------------------------------------------------------------------------
constexpr int PGR_ONE_NT = 1024;

int pgr_update_blocks(long n, int m, int nb)
{
    if (m > MAXM_FAST) return nb;
    const long g = ((n + 1) / 2 + PGR_ONE_NT - 1) / PGR_ONE_NT;
    return (int)std::max(1L, g);
}

template <typename T, int MM, int NT, bool ONE>
__global__ __launch_bounds__(NT) void pgr_update_kernel(const PUpdArgs<T> a)
{
    constexpr int NS = MM + 1;
    __shared__ double scratch[NT / 64];
    __shared__ double sums[1];
    if (a.ctrl->done) return;
    const int nv = a.nvalid;
    const T *px[NS], *py[NS];
    bool use[NS];
    T sv[MM];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        use[k] = k <= nv;
        const size_t off = (size_t)(use[k] ? a.slot[k] : 0) * a.ld;
        px[k] = a.X + off;
        py[k] = a.Y + off;
    }
#pragma unroll
    for (int k = 0; k < MM; k++) sv[k] = k < nv ? (T)a.ctrl->s[ref_col(a.it, k, a.m, 0)] : (T)0;
    T *xc = a.X + (size_t)a.slot[0] * a.ld;
    T *yc = a.Y + (size_t)a.slot[0] * a.ld;
    double acc[1] = {0.0};

    T *xn = a.next >= 0 ? a.X + (size_t)a.next * a.ld : nullptr;
    const T om = (T)a.omega, dg = (T)a.diag;
    // PGR.c:92-98 at a point with f = b - Ax and the divisor d
    auto rich = [&](T xv, T f, T d) -> T {
        if (a.precond) f = f / d;
        return xv + om * f;
    };

    auto point = [&](const T (&vx)[NS], const T (&vy)[NS], T &xv, T &yv) {
        xv = vx[0];
        yv = vy[0];
#pragma unroll
        for (int k = 0; k < MM; k++) {
            if (k < nv) {
                xv = xv + (vx[k] - vx[k + 1]) * sv[k];
                yv = yv + (vy[k] - vy[k + 1]) * sv[k];
            }
        }
    };

    const long n = a.n;
    const long stride = (long)gridDim.x * NT;
    if ((n & 1) == 0) {
        using V2 = typename Vec2<T>::type;
        const long np = n >> 1;
        for (long ip = ONE ? (long)blockIdx.x * NT + threadIdx.x : chunk_first(); ip < np;
             ip = ONE ? np : chunk_next(ip)) {
            const long i = 2 * ip;
            T vx0[NS], vx1[NS], vy0[NS], vy1[NS];
#pragma unroll
            for (int k = 0; k < NS; k++) {
                vx0[k] = vx1[k] = vy0[k] = vy1[k] = (T)0;
                if (use[k]) {
                    const V2 u = ld_nt2<V2>(px[k] + i);
                    const V2 w = ld_nt2<V2>(py[k] + i);
                    vx0[k] = u.x;
                    vx1[k] = u.y;
                    vy0[k] = w.x;
                    vy1[k] = w.y;
                }
            }
            V2 xo, yo;
            point(vx0, vy0, xo.x, yo.x);
            point(vx1, vy1, xo.y, yo.y);
            st_nt2(xc + i, xo);
            st_nt2(yc + i, yo);
            const V2 bv = ld_nt2<V2>(a.b + i);
            const T r0 = bv.x - yo.x, r1 = bv.y - yo.y;            // PGR.c:129-130
            acc[0] += (double)r0 * (double)r0;
            acc[0] += (double)r1 * (double)r1;
            if (xn) {
                T d0 = dg, d1 = dg;
                if (a.c) {
                    d0 = dg + a.c[i];
                    d1 = dg + a.c[i + 1];
                }
                V2 no;
                no.x = rich(xo.x, r0, d0);
                no.y = rich(xo.y, r1, d1);
                st_nt2(xn + i, no);
            }
        }
    } else {
        for (long i = (long)blockIdx.x * NT + threadIdx.x; i < n; i += stride) {
            T vx[NS], vy[NS];
#pragma unroll
            for (int k = 0; k < NS; k++) {
                vx[k] = use[k] ? px[k][i] : (T)0;
                vy[k] = use[k] ? py[k][i] : (T)0;
            }
            T xv, yv;
            point(vx, vy, xv, yv);
            xc[i] = xv;
            yc[i] = yv;
            const T r = a.b[i] - yv;
            acc[0] += (double)r * (double)r;
            if (xn) xn[i] = rich(xv, r, a.c ? dg + a.c[i] : dg);
        }
    }
    block_reduce_to<1, NT>(acc, a.partials + blockIdx.x, scratch);
    if (!a.counter) return;                     // two-pass: finish_kernel follows
    if (last_block_arrive(a.counter, gridDim.x)) {
        final_sum<NT>(a.partials, a.nblocks, 1, sums, scratch);
        if (threadIdx.x == 0) {
            finalize(a.fin, a.ctrl, sums, 1);
            *a.counter = 0u;
        }
    }
}

template <typename T>
hipError_t launch_pgr_update(const PUpdArgs<T> &a, hipStream_t st)
{
    if (a.m < 1 || a.m > MAXM || a.nvalid < 0 || a.nvalid > a.m) return hipErrorInvalidValue;
    // the grid is the caller's partial count: pgr_update_blocks()
    if (a.m <= MAXM_FAST && a.nblocks != pgr_update_blocks(a.n, a.m, a.nblocks)) return hipErrorInvalidValue;
    if (a.m <= MAXM_FAST)
        hipLaunchKernelGGL((pgr_update_kernel<T, MAXM_FAST, PGR_ONE_NT, true>), dim3(a.nblocks), dim3(PGR_ONE_NT), 0,
                           st, a);
    else if (a.m <= MAXM_MID)
        hipLaunchKernelGGL((pgr_update_kernel<T, MAXM_MID, BLOCK, false>), dim3(a.nblocks), dim3(BLOCK), 0, st, a);
    else hipLaunchKernelGGL((pgr_update_kernel<T, MAXM, BLOCK, false>), dim3(a.nblocks), dim3(BLOCK), 0, st, a);
    return hipGetLastError();
}
template hipError_t launch_pgr_update<double>(const PUpdArgs<double> &, hipStream_t);
template hipError_t launch_pgr_update<float>(const PUpdArgs<float> &, hipStream_t);

// ---------------------------------------------------------------------------
// dots and CG pointwise step
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(BLOCK) void dot_kernel(const DotArgs<T> a)
{
    __shared__ double scratch[BLOCK / 64];
    __shared__ double sums[1];
    if (a.ctrl->done) return;
    double acc[1] = {0.0};
    const T *w = a.w ? a.w : a.v;
    const long stride = (long)gridDim.x * BLOCK;
    for (long i = chunk_first(); i < a.n; i = chunk_next(i))
        acc[0] += (double)a.v[i] * (double)w[i];
    block_reduce_to<1>(acc, a.partials + blockIdx.x, scratch);
    if (!a.counter) return;                     // two-pass: finish_kernel follows
    if (last_block_arrive(a.counter, gridDim.x)) {
        final_sum(a.partials, a.nblocks, 1, sums, scratch);
        if (threadIdx.x == 0) {
            finalize(a.fin, a.ctrl, sums, 1);
            *a.counter = 0u;
        }
    }
}

template <typename T>
hipError_t launch_dot(const DotArgs<T> &a, hipStream_t st)
{
    hipLaunchKernelGGL((dot_kernel<T>), dim3(a.nblocks), dim3(BLOCK), 0, st, a);
    return hipGetLastError();
}
template hipError_t launch_dot<double>(const DotArgs<double> &, hipStream_t);
template hipError_t launch_dot<float>(const DotArgs<float> &, hipStream_t);

// The pointwise steps of CG.  One pair per thread and one block (and one
// pair of partials) per CG_NT pairs, every stream non-temporal.  Odd n, or a
// vector off a 16-byte boundary, walks a grid stride element by element over
// the same grid with the same arithmetic.
constexpr int CG_NT = 1024;

int cg_blocks(long n)
{
    const long g = ((n + 1) / 2 + CG_NT - 1) / CG_NT;
    return (int)std::max(1L, g);
}

// the element arithmetic; x is updated when HX
template <CgStep S, bool HX>
__device__ __forceinline__ void cg_point(const CgArgs &a, double alpha, double beta, double dg, double &x, double &r,
                                         double &d, double q, double (&acc)[2])
{
    if (HX) x = x + alpha * d;                          // CG.c:106-107
    if (S == CgStep::DIR || S == CgStep::RES) {
        if (S == CgStep::RES) r = r - alpha * q;        // CG.c:121-124
        double s = r;
        if (a.precond) s = s / dg;
        if (S == CgStep::DIR) {
            d = s + beta * d;                           // CG.c:148-150
        } else {
            acc[0] += r * s;
            acc[1] += r * r;
        }
    }
}

template <CgStep S, bool HX>
__global__ __launch_bounds__(CG_NT) void cg_kernel(const CgArgs a)
{
    constexpr int NT = CG_NT;
    constexpr bool RD = S == CgStep::DIR || S == CgStep::RES;      // the steps on r
    constexpr bool HD = HX || S == CgStep::DIR;                    // reads d
    __shared__ double scratch[2 * (NT / 64)];
    __shared__ double sums[2];
    if (S == CgStep::X_PENDING) {
        if (!a.ctrl->xpend) return;
    } else if (a.ctrl->done) {
        return;
    }
    const double alpha = a.ctrl->alpha, beta = a.ctrl->beta;
    double acc[2] = {0.0, 0.0};
    const long n = a.n;
    const uintptr_t al = (HX ? (uintptr_t)a.x : 0) | (RD ? (uintptr_t)a.r : 0) | (HD ? (uintptr_t)a.d : 0) |
                         (S == CgStep::RES ? (uintptr_t)a.q : 0) | (RD && a.c ? (uintptr_t)a.c : 0);
    if ((n & 1) == 0 && al % 16 == 0) {
        using V2 = typename Vec2<double>::type;
        const long ip = (long)blockIdx.x * NT + threadIdx.x;
        if (ip < (n >> 1)) {
            const long i = 2 * ip;
            V2 x = {}, r = {}, d = {}, q = {};
            if (HX) x = ld_nt2<V2>(a.x + i);
            if (RD) r = ld_nt2<V2>(a.r + i);
            if (HD) d = ld_nt2<V2>(a.d + i);
            if (S == CgStep::RES) q = ld_nt2<V2>(a.q + i);
            double d0 = a.diag, d1 = a.diag;
            if (RD && a.c) {
                const V2 cv = ld_nt2<V2>(a.c + i);
                d0 = a.diag + cv.x;
                d1 = a.diag + cv.y;
            }
            cg_point<S, HX>(a, alpha, beta, d0, x.x, r.x, d.x, q.x, acc);
            cg_point<S, HX>(a, alpha, beta, d1, x.y, r.y, d.y, q.y, acc);
            if (HX) st_nt2(a.x + i, x);
            if (S == CgStep::RES) st_nt2(a.r + i, r);
            if (S == CgStep::DIR) st_nt2(a.d + i, d);
        }
    } else {
        for (long i = (long)blockIdx.x * NT + threadIdx.x; i < n; i += (long)gridDim.x * NT) {
            double x = HX ? a.x[i] : 0.0, r = RD ? a.r[i] : 0.0, d = HD ? a.d[i] : 0.0;
            cg_point<S, HX>(a, alpha, beta, RD && a.c ? a.diag + a.c[i] : a.diag, x, r, d,
                            S == CgStep::RES ? a.q[i] : 0.0, acc);
            if (HX) a.x[i] = x;
            if (S == CgStep::RES) a.r[i] = r;
            if (S == CgStep::DIR) a.d[i] = d;
        }
    }
    if (S != CgStep::RES) return;
    block_reduce_to<2, NT>(acc, a.partials + (size_t)blockIdx.x * 2, scratch);
    if (!a.counter) return;                     // two-pass: finish_kernel follows
    if (last_block_arrive(a.counter, gridDim.x)) {
        final_sum<NT>(a.partials, a.nblocks, 2, sums, scratch);
        if (threadIdx.x == 0) {
            finalize(a.fin, a.ctrl, sums, 2);
            *a.counter = 0u;
        }
    }
}

hipError_t launch_cg(CgStep step, const CgArgs &a, hipStream_t st)
{
    // the grid is the caller's partial count: cg_blocks()
    if (a.nblocks != cg_blocks(a.n)) return hipErrorInvalidValue;
    if (step != CgStep::DIR && step != CgStep::RES && !a.x) return hipErrorInvalidValue;
    const dim3 grid(a.nblocks), block(CG_NT);
    switch (step) {
    case CgStep::DIR:
        if (a.x) hipLaunchKernelGGL((cg_kernel<CgStep::DIR, true>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((cg_kernel<CgStep::DIR, false>), grid, block, 0, st, a);
        break;
    case CgStep::RES: hipLaunchKernelGGL((cg_kernel<CgStep::RES, false>), grid, block, 0, st, a); break;
    case CgStep::X: hipLaunchKernelGGL((cg_kernel<CgStep::X, true>), grid, block, 0, st, a); break;
    case CgStep::X_PENDING: hipLaunchKernelGGL((cg_kernel<CgStep::X_PENDING, true>), grid, block, 0, st, a); break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// second pass of a reduction: one block sums per-block partials in a fixed
// order and runs the finaliser (no device-scope fence or atomic needed: the
// kernel boundary orders it after the partials); further blocks sum the
// recorded norms (TraceFin).  A launch is a chain of latencies, 2.8-4.6 us
// whatever it sums: one per check instead of one per sweep takes AAR at
// 48^3 from 6.48 to 5.74 ms, complex AAR with gradients at 96^3 28.8 -> 27.4.
// A record does not wait for `done`: block 0 may set it meanwhile, and what a
// sweep skipped after convergence leaves lies past the history that is read.
// ---------------------------------------------------------------------------
template <int NT, int NACC>
__global__ __launch_bounds__(NT) void finish_kernel(const double *partials, int nitems, FinArgs fin, Ctrl *ctrl,
                                                    const TraceFin tr)
{
    __shared__ double scratch[NACC * (NT / 64)];
    __shared__ double sums[NACC];
    if (blockIdx.x > 0) {
        const int j = blockIdx.x - 1, i = tr.it0 - 1 + j;
        final_sum<NT>(tr.partials + (size_t)j * tr.nitems, tr.nitems, 1, sums, scratch);
        if (threadIdx.x == 0 && i >= 0 && i < tr.hist_cap) tr.hist[i] = sqrt(sums[0]);
        return;
    }
    if (!partials || ctrl->done) return;
    // every value's sum in one pass, in final_sum's order
    double acc[NACC];
#pragma unroll
    for (int k = 0; k < NACC; k++) acc[k] = 0.0;
#pragma unroll 4
    for (int i = threadIdx.x; i < nitems; i += NT)
#pragma unroll
        for (int k = 0; k < NACC; k++) acc[k] += partials[(size_t)i * NACC + k];
#pragma unroll
    for (int k = 0; k < NACC; k++) {
        acc[k] = wave_sum(acc[k]);
        if ((threadIdx.x & 63) == 0) scratch[k * (NT / 64) + (threadIdx.x >> 6)] = acc[k];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int k = 0; k < NACC; k++) {
        double t = 0.0;
        for (int w = 0; w < NT / 64; w++) t += scratch[k * (NT / 64) + w];
        sums[k] = t;
    }
    finalize(fin, ctrl, sums, NACC);
}

hipError_t launch_finish(const double *partials, int nitems, int nacc, const FinArgs &fin, Ctrl *ctrl,
                         hipStream_t st, const TraceFin &tr)
{
    if (nacc < 1 || nacc > 2) return hipErrorInvalidValue;
    const dim3 grid(1 + tr.count);
    // sixteen wavefronts once four would walk more than a few dozen partials
    // each (CG at 250 x 256 x 243, 7594 pairs a residual: 369 -> 356 ms)
    auto go = [&](auto nt, auto na) {
        constexpr int NT = decltype(nt)::value, NA = decltype(na)::value;
        hipLaunchKernelGGL((finish_kernel<NT, NA>), grid, dim3(NT), 0, st, partials, nitems, fin, ctrl, tr);
    };
    using std::integral_constant;
    const bool big = nitems > 2048;
    if (nacc == 1 && !big) go(integral_constant<int, BLOCK>{}, integral_constant<int, 1>{});
    else if (nacc == 1) go(integral_constant<int, 1024>{}, integral_constant<int, 1>{});
    else if (!big) go(integral_constant<int, BLOCK>{}, integral_constant<int, 2>{});
    else go(integral_constant<int, 1024>{}, integral_constant<int, 2>{});
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__global__ void copy_f64_kernel(double *dst, const double *src, long n, const Ctrl *c)
{
    if (c && c->done) return;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}
template <typename T>
__global__ void fill_kernel(T *dst, T v, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        dst[i] = v;
}
__global__ void axpy_f64_f32_kernel(double *x, const float *e, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        x[i] = x[i] + (double)e[i];
}
__global__ void div_f64_kernel(double *r, double d, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        r[i] /= d;
}
__global__ void zero_ctrl_kernel(Ctrl *c)
{
    double *p = reinterpret_cast<double *>(c);
    const int nw = (int)(sizeof(Ctrl) / sizeof(double));
    for (int i = threadIdx.x; i < nw; i += blockDim.x) p[i] = 0.0;
}

static unsigned grid_for(long n)
{
    long g = (n + BLOCK - 1) / BLOCK;
    return (unsigned)(g > 8192 ? 8192 : (g < 1 ? 1 : g));
}

hipError_t launch_copy_f64(double *dst, const double *src, long n, const Ctrl *ctrl, hipStream_t st)
{
    hipLaunchKernelGGL(copy_f64_kernel, dim3(grid_for(n)), dim3(BLOCK), 0, st, dst, src, n, ctrl);
    return hipGetLastError();
}
hipError_t launch_fill_f64(double *dst, double v, long n, hipStream_t st)
{
    hipLaunchKernelGGL((fill_kernel<double>), dim3(grid_for(n)), dim3(BLOCK), 0, st, dst, v, n);
    return hipGetLastError();
}
hipError_t launch_fill_f32(float *dst, float v, long n, hipStream_t st)
{
    hipLaunchKernelGGL((fill_kernel<float>), dim3(grid_for(n)), dim3(BLOCK), 0, st, dst, v, n);
    return hipGetLastError();
}
hipError_t launch_axpy_f64_f32(double *x, const float *e, long n, hipStream_t st)
{
    hipLaunchKernelGGL(axpy_f64_f32_kernel, dim3(grid_for(n)), dim3(BLOCK), 0, st, x, e, n);
    return hipGetLastError();
}
hipError_t launch_div_f64(double *r, double diag, long n, hipStream_t st)
{
    hipLaunchKernelGGL(div_f64_kernel, dim3(grid_for(n)), dim3(BLOCK), 0, st, r, diag, n);
    return hipGetLastError();
}
hipError_t launch_zero_ctrl(Ctrl *c, hipStream_t st)
{
    hipLaunchKernelGGL(zero_ctrl_kernel, dim3(1), dim3(256), 0, st, c);
    return hipGetLastError();
}

}  // namespace aar
