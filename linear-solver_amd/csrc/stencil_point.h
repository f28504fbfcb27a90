// stencil_point.h -- what the two forms of the FD12 stencil sweep share: the
// lane layout, the memory accesses, the operator at a row of points and the
// epilogue of each mode (see stencil.hip for the design notes).
#pragma once

#include <type_traits>

#include "aar_common.h"
#include "aar_device.h"
#include "aar_kernels.h"

namespace aar {

template <typename T> struct Arith;
template <> struct Arith<double> {
    __device__ static inline double add(double a, double b) { return __dadd_rn(a, b); }
    __device__ static inline double sub(double a, double b) { return __dsub_rn(a, b); }
    __device__ static inline double mul(double a, double b) { return __dmul_rn(a, b); }
    __device__ static inline double div(double a, double b) { return a / b; }
    __device__ static inline double sq(double a) { return a * a; }
};
template <> struct Arith<float> {
    __device__ static inline float add(float a, float b) { return __fadd_rn(a, b); }
    __device__ static inline float sub(float a, float b) { return __fsub_rn(a, b); }
    __device__ static inline float mul(float a, float b) { return __fmul_rn(a, b); }
    __device__ static inline float div(float a, float b) { return __fdiv_rn(a, b); }
    __device__ static inline double sq(float a) { return (double)a * (double)a; }
};

// NE: epilogue inputs besides the coefficient field; NACC: norm sums
template <SMode M> struct ModeInfo {
    static constexpr int NE = M == SMode::MATVEC || M == SMode::AAR_REC || M == SMode::CG_Q ? 0 : 1;
    static constexpr int NACC = M == SMode::CG_RESID ? 2 : 1;
};

__device__ inline int modp(int i, int n) { i %= n; return i < 0 ? i + n : i; }

// Lane layout: a lane owns V consecutive x-points (16 bytes), so that the
// plane tile in LDS is read and written 16 bytes a lane.  On gfx950 that
// streams 200 B/clk per CU against 115 (8-byte) and 70 (4-byte accesses),
// and the x-neighbours of V points share their loads: an FP64 point takes 17
// doubles from LDS (one point a lane: 21), an FP32 point 16 floats.  A tile
// row of TX = 64 points is LPR lanes, a wavefront covers RPW rows.  HXV
// vectors of x-halo on each side cover the radius.
template <typename T> struct Lane {
    static constexpr int V = 16 / (int)sizeof(T);
    static constexpr int LPR = TX / V;
    static constexpr int RPW = 64 / LPR;
    static constexpr int HXV = (R + V - 1) / V;
    static constexpr int LW = TX + 2 * HXV * V;        // row pitch of the plane tile
    typedef T Vec __attribute__((ext_vector_type(V)));
    // the same in global memory: rows start at multiples of nx, the caller's
    // vectors at any element (gfx950 takes 16-byte accesses at any dword)
    typedef T VecU __attribute__((ext_vector_type(V), aligned(sizeof(T))));
};

// Width of a one-shot box of lz planes.  FP64 boxes of 2 and 4 planes are 32 x
// 16 points: 1.1 halo values a point against 1.7 of 64 x 8, and less of a tile
// past an x-side (recurrence sweep with a one-vector update, 64 wide / 32: 96^3
// 16.9 / 15.4 us, 160^3 48.3 / 44.3, 200^3 93.2 / 88.6; PGR at 128^3 103.5 ->
// 99.8 ms).  One plane: 64 x 8 (AAR at 48^3 5.80 ms, 32 wide 5.87).  FP32 64 x
// 16 (32 x 32: 200 x 161 x 150 32.1 -> 32.9 us, 96^3 14.4 -> 13.7).
template <typename T> __host__ __device__ constexpr int tile_x(int lz) { return sizeof(T) == 8 && lz > 1 ? 32 : 64; }

// How the tiles of a grid take their vectors of V points along x, chosen at
// launch (x_mode), a kernel each, so that no grid pays for the registers of
// another's form.
// * XVEC (nx a multiple of V): the V points are consecutive in memory, one
//   access and one offset.
// * XSHIFT (any other nx from a tile and its halo up): tiles that would reach
//   past nx, or whose halo would, start earlier instead (tile_x0), so that no
//   vector wraps inside: the same accesses, at any alignment of a row.  Points
//   covered by two tiles are computed twice, by the same operations; the norms
//   take them once.  With the tiles at the end of a row point by point (20
//   accesses for 5), an iteration of the mixed solve took 84 us at 193 x 189 x 196
//   against 57, the FP32 operator 454 against 274 at 449 x 445 x 452.
// * XPOINT (narrower grids, down to which the march narrows its columns first:
//   march_width): point by point, a wrapped offset each.
// * XWIDE: the same with 64-bit byte offsets, for the planes of wide_plane().
enum : int { XVEC = 0, XSHIFT = 1, XPOINT = 2, XWIDE = 3 };

// Byte offsets in a plane are 32 bits wide.  A plane of more than 2^32 bytes
// (2^29 points FP64, 2^30 FP32) takes the XWIDE sweep.
template <typename T> __host__ __device__ inline bool wide_plane(int nx, int ny)
{
    return (unsigned long long)nx * (unsigned long long)ny * sizeof(T) > 1ull << 32;
}

// base[off] with a uniform (per-plane) base pointer and a 32-bit in-plane
// offset: the access compiles to the scalar-base + vector-offset form, with
// no per-access 64-bit address arithmetic
template <typename T, bool WIDE> __device__ __forceinline__ size_t byte_off(unsigned eoff)
{
    if constexpr (WIDE) return (size_t)eoff * sizeof(T);
    else return (size_t)(eoff * (unsigned)sizeof(T));
}
template <bool WIDE, typename T> __device__ __forceinline__ T ld_at(const T *base, unsigned eoff)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte_off<T, WIDE>(eoff));
}
template <bool WIDE, typename T> __device__ __forceinline__ void st_at(T *base, unsigned eoff, T v)
{
    *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + byte_off<T, WIDE>(eoff)) = v;
}

// in-plane element offsets of one vector of points
template <typename T, int XM> struct VOff {
    static constexpr int NO = XM <= XSHIFT ? 1 : Lane<T>::V;
    unsigned o[NO];
    __device__ __forceinline__ void set(int gx, int gy, int nx, int ny)
    {
        const int row = modp(gy, ny) * nx;
#pragma unroll
        for (int v = 0; v < NO; v++) o[v] = (unsigned)(row + modp(gx + v, nx));
    }
};

template <typename T, int XM>
__device__ __forceinline__ typename Lane<T>::Vec ld_vec(const T *base, const VOff<T, XM> &f)
{
    using L = Lane<T>;
    typename L::Vec r;
    if constexpr (XM <= XSHIFT) {
        r = *reinterpret_cast<const typename L::VecU *>(reinterpret_cast<const char *>(base) +
                                                        (size_t)(f.o[0] * (unsigned)sizeof(T)));
    } else {
#pragma unroll
        for (int v = 0; v < L::V; v++) r[v] = ld_at<XM == XWIDE>(base, f.o[v]);
    }
    return r;
}

// How tiles w wide take the vectors of a grid
template <typename T> __host__ __device__ inline int x_mode(int nx, int ny, int w)
{
    using L = Lane<T>;
    if (wide_plane<T>(nx, ny)) return XWIDE;
    if (nx % L::V == 0) return XVEC;
    return nx >= w + L::HXV * L::V ? XSHIFT : XPOINT;
}

// First point x0 of the W-wide tile itx, and the first one whose norm terms are
// its own.  XSHIFT: the last tile ends at nx, and the one before it a halo short
// of nx where its halo would wrap inside a vector.
template <typename T, int W, int XM>
__device__ __forceinline__ void tile_x0(int itx, int nx, int &x0, int &own)
{
    constexpr int HX = Lane<T>::HXV * Lane<T>::V;
    x0 = own = itx * W;
    if constexpr (XM == XSHIFT) {
        if (nx % Lane<T>::V == 0) return;
        if (x0 + W >= nx) {
            own = x0 + HX > nx ? nx - HX : x0;        // where the tile before it ends
            x0 = nx - W;
        } else if (x0 + W + HX > nx) {
            x0 = nx - HX - W;
        }
    }
}

// S: the stored type (T, or float for the FP32 copy of an FP64 sweep).
// NT: non-temporal.  ok: masks of the V points, or of the vector (ok[0]).
template <typename S, bool NT, typename T, int XM, int NV>
__device__ __forceinline__ void st_vec(S *base, const VOff<T, XM> &f, const S (&v)[NV], const bool (&ok)[NV],
                                       bool masked)
{
    if constexpr (XM <= XSHIFT) {
        typedef S SV __attribute__((ext_vector_type(NV), aligned(sizeof(S))));
        SV r;
#pragma unroll
        for (int i = 0; i < NV; i++) r[i] = v[i];
        SV *p = reinterpret_cast<SV *>(reinterpret_cast<char *>(base) + (size_t)(f.o[0] * (unsigned)sizeof(S)));
        if (!masked || ok[0]) {
            if constexpr (NT) __builtin_nontemporal_store(r, p);
            else *p = r;
        }
    } else {
#pragma unroll
        for (int i = 0; i < NV; i++)
            if (!masked || ok[i]) st_at<XM == XWIDE>(base, f.o[i], v[i]);
    }
}

// per-launch constants of the point formulas
template <typename T> struct PointK {
    T wt[R + 1], cf[R + 1], sig, dg, om, w3;
    double trace_scale;
    __device__ __forceinline__ explicit PointK(const SArgs<T> &a)
    {
#pragma unroll
        for (int o = 0; o <= R; o++) wt[o] = (T)a.w[o];
        sig = (T)a.sigma;
        dg = (T)a.diag;
        om = (T)a.omega;
        w3 = (T)(3.0 * a.w[0]);
#pragma unroll
        for (int o = 0; o <= R; o++) cf[o] = (T)a.cf[o];
        trace_scale = a.precond ? a.diag : 1.0;
    }
};

// The operator at V consecutive points: xw the x-window (own points from
// index HXV*V), yn(d), zn(d) the vectors d rows / planes away, vv the
// pointwise field (VC).  system.c:195-201 order: centre, then o = 1..6 with
// (x-, x+, y-, y+, z-, z+) summed left to right.
template <typename T, SMode MODE, bool VC, typename YN, typename ZN>
__device__ __forceinline__ typename Lane<T>::Vec stencil_value(const SArgs<T> &a, const PointK<T> &k,
                                                               const T (&xw)[(2 * Lane<T>::HXV + 1) * Lane<T>::V],
                                                               const typename Lane<T>::Vec vv, YN yn, ZN zn)
{
    using A = Arith<T>;
    using L = Lane<T>;
    using Vec = typename L::Vec;
    constexpr int V = L::V, C = L::HXV * V;
    Vec y;
    // the six neighbours at distance o of point v
    auto nb6 = [&](int o, int v, const Vec &ym, const Vec &yp, const Vec &zm, const Vec &zp) -> T {
        T nb = A::add(xw[C + v - o], xw[C + v + o]);
        nb = A::add(nb, ym[v]);
        nb = A::add(nb, yp[v]);
        nb = A::add(nb, zm[v]);
        return A::add(nb, zp[v]);
    };
    if constexpr (MODE == SMode::AAR_REC && VC) {
        // variable coefficient, D = diag + c(x): A g = D g +
        // sum_o w_o S_o, so with the Jacobi step g' = g -
        // (omega/D) A g = (1 - omega) g - h sum_o w_o S_o, h =
        // omega/D = a.vf; without a preconditioner a.vf = c and
        // g' = (1 - omega (3 w0 + c)) g - omega sum_o w_o S_o
        Vec ns;
#pragma unroll
        for (int v = 0; v < V; v++) ns[v] = (T)0;
#pragma unroll
        for (int o = 1; o <= R; o++) {
            const Vec ym = yn(-o), yp = yn(o), zm = zn(-o), zp = zn(o);
#pragma unroll
            for (int v = 0; v < V; v++) ns[v] = fma(nb6(o, v, ym, yp, zm, zp), k.wt[o], ns[v]);
        }
#pragma unroll
        for (int v = 0; v < V; v++) {
            const T u = xw[C + v];
            if (a.precond) y[v] = fma(-vv[v], ns[v], A::mul(u, k.cf[0]));
            else y[v] = fma(-k.om, ns[v], A::mul(u, A::sub((T)1, A::mul(k.om, A::add(k.w3, vv[v])))));
        }
    } else if constexpr (MODE == SMode::AAR_REC) {
        // the Richardson step folded into the weights: g' = cf0 g +
        // sum_o cf_o S_o, cf0 = 1 - c (3 w0 + sigma), cf_o = -c w_o,
        // c = omega/diag (no reference counterpart; the reference
        // recomputes b - A x, see the solver)
#pragma unroll
        for (int v = 0; v < V; v++) y[v] = A::mul(xw[C + v], k.cf[0]);
#pragma unroll
        for (int o = 1; o <= R; o++) {
            const Vec ym = yn(-o), yp = yn(o), zm = zn(-o), zp = zn(o);
#pragma unroll
            for (int v = 0; v < V; v++) y[v] = fma(nb6(o, v, ym, yp, zm, zp), k.cf[o], y[v]);
        }
    } else if constexpr (sizeof(T) == 8) {
#pragma unroll
        for (int v = 0; v < V; v++) y[v] = A::mul(A::mul(xw[C + v], (T)3), k.wt[0]);
#pragma unroll
        for (int o = 1; o <= R; o++) {
            const Vec ym = yn(-o), yp = yn(o), zm = zn(-o), zp = zn(o);
#pragma unroll
            for (int v = 0; v < V; v++) y[v] = A::add(y[v], A::mul(nb6(o, v, ym, yp, zm, zp), k.wt[o]));
        }
    } else {
        // FP32 (no reference counterpart): difference form
        // sum_o w_o * sum_nb (x_nb - x_c), i.e. the centre weight taken
        // as -2 sum_o w_o.  Row sums are exactly zero and each rounding
        // is relative to a local difference, so the smooth modes, whose
        // eigenvalues are tiny, keep their accuracy; the reference form
        // would shift them by ~eps32 * |w_0| and stall FP32 iterations.
#pragma unroll
        for (int v = 0; v < V; v++) y[v] = (T)0;
#pragma unroll
        for (int o = 1; o <= R; o++) {
            const Vec ym = yn(-o), yp = yn(o), zm = zn(-o), zp = zn(o);
#pragma unroll
            for (int v = 0; v < V; v++) {
                const T u = xw[C + v];
                T nb = A::add(A::sub(xw[C + v - o], u), A::sub(xw[C + v + o], u));
                nb = A::add(nb, A::sub(ym[v], u));
                nb = A::add(nb, A::sub(yp[v], u));
                nb = A::add(nb, A::sub(zm[v], u));
                nb = A::add(nb, A::sub(zp[v], u));
                y[v] = A::add(y[v], A::mul(nb, k.wt[o]));
            }
        }
    }
    if constexpr (MODE != SMode::AAR_REC) {
        if (a.sigma != 0.0) {
#pragma unroll
            for (int v = 0; v < V; v++) y[v] = A::add(y[v], A::mul(k.sig, xw[C + v]));
        }
        // y + c(x) x, the order of the screened term above
        if constexpr (VC) {
#pragma unroll
            for (int v = 0; v < V; v++) y[v] = A::add(y[v], A::mul(vv[v], xw[C + v]));
        }
    }
    return y;
}

// What a sweep does with y = A u at V points: its outputs through
// put(base, values) and its norm terms into acc.  Points past the grid edge
// (partial tiles) are computed on wrapped inputs.  Such a lane reads exactly
// what the lane owning the wrapped point reads, through the same operations,
// so it may store the same bits to the same address: put may store
// unconditionally (no branch per point) or masked.  Norm terms are always
// masked, per vector in XVEC, else per point.
template <typename T, SMode MODE, bool VC, int XM, int NACC, typename Put>
__device__ __forceinline__ void stencil_epilogue(const SArgs<T> &a, const PointK<T> &k,
                                                 const typename Lane<T>::Vec y, const typename Lane<T>::Vec u,
                                                 const typename Lane<T>::Vec en, const typename Lane<T>::Vec vv,
                                                 const bool (&ok)[Lane<T>::V], Put put, double (&acc)[NACC])
{
    using A = Arith<T>;
    constexpr int V = Lane<T>::V;
    T o0[V], o1[V];
    float of[V];
    double t[NACC];
#pragma unroll
    for (int j = 0; j < NACC; j++) t[j] = 0.0;
    auto m = [&](int v, double x) -> double {
        if constexpr (XM != XVEC) return ok[v] ? x : 0.0;
        else return x;
    };
    if constexpr (MODE == SMode::MATVEC) {
#pragma unroll
        for (int v = 0; v < V; v++) o0[v] = y[v];
        put(a.out0, o0);
    } else if constexpr (MODE == SMode::AAR_TRUE) {
        // AAR.c:80-82/93-94/119-123: f = (rhs - A x)/diag, stored in
        // T or (mixed precision) rounded to FP32; ||rhs - A x||^2
#pragma unroll
        for (int v = 0; v < V; v++) {
            const T r = A::sub(en[v], y[v]);
            t[0] += m(v, A::sq(r));
            T f = r;
            if constexpr (VC) {
                if (a.precond) f = A::div(f, A::add(k.dg, vv[v]));
            } else {
                if (a.precond) f = A::div(f, k.dg);
            }
            o0[v] = f;
            of[v] = (float)f;
        }
        if (a.out32) put(a.out32, of);
        else put(a.out0, o0);
    } else if constexpr (MODE == SMode::AAR_REC) {
        // y = g_{k+1} = (rhs - A(x_k + omega g_k))/diag; scale^2 *
        // ||g_{k+1}||^2 = ||rhs - A x_{k+1}||^2 for the history
#pragma unroll
        for (int v = 0; v < V; v++) o0[v] = y[v];
        put(a.out0, o0);
        if (a.trace) {
#pragma unroll
            for (int v = 0; v < V; v++) {
                // ||rhs - A x||: D g' pointwise (VC: D = omega/h, by
                // the hardware reciprocal -- the trace is a record,
                // convergence is decided on the AAR_TRUE sweep)
                double sv;
                if constexpr (VC)
                    sv = (double)y[v] * (a.precond ? a.omega * __builtin_amdgcn_rcp((double)vv[v]) : 1.0);
                else
                    sv = (double)y[v] * k.trace_scale;
                sv = m(v, sv);
                t[0] = fma(sv, sv, t[0]);
            }
        }
    } else if constexpr (MODE == SMode::RESID) {
#pragma unroll
        for (int v = 0; v < V; v++) {
            const T r = A::sub(en[v], y[v]);
            t[0] += m(v, A::sq(r));
            o0[v] = r;
            of[v] = (float)r;
        }
        if (a.out32) put(a.out32, of);
        if (a.out0) put(a.out0, o0);
    } else if constexpr (MODE == SMode::PGR_STEP) {
        // PGR.c:92-103: Ax = A x; f = rhs - Ax; the next iterate is
        // x + omega f / diag, pointwise
#pragma unroll
        for (int v = 0; v < V; v++) {
            T f = A::sub(en[v], y[v]);
            t[0] += m(v, A::sq(f));
            if constexpr (VC) {
                if (a.precond) f = A::div(f, A::add(k.dg, vv[v]));
            } else {
                if (a.precond) f = A::div(f, k.dg);
            }
            o0[v] = y[v];
            o1[v] = A::add(u[v], A::mul(k.om, f));
        }
        put(a.out0, o0);
        if (a.out1) put(a.out1, o1);
    } else if constexpr (MODE == SMode::CG_Q) {
        // CG.c:94-100: q = A d; alpha partial d.q
#pragma unroll
        for (int v = 0; v < V; v++) {
            o0[v] = y[v];
            t[0] += m(v, (double)u[v] * (double)y[v]);
        }
        put(a.out0, o0);
    } else if constexpr (MODE == SMode::CG_RESID) {
        // CG.c:65-84 / 112-119: r = b - A x; s = r/diag; r.s, r.r
#pragma unroll
        for (int v = 0; v < V; v++) {
            const T r = A::sub(en[v], y[v]);
            T s = r;
            if constexpr (VC) {
                if (a.precond) s = A::div(s, A::add(k.dg, vv[v]));
            } else {
                if (a.precond) s = A::div(s, k.dg);
            }
            o0[v] = r;
            o1[v] = s;
            t[0] += m(v, (double)r * (double)s);
            t[1] += m(v, A::sq(r));
        }
        put(a.out0, o0);
        if (a.out1) put(a.out1, o1);
    }
#pragma unroll
    for (int j = 0; j < NACC; j++) acc[j] += XM != XVEC || ok[0] ? t[j] : 0.0;
}

}  // namespace aar
