// ls_body.h -- the m x m pseudo-inverse solve of the Anderson, Galerkin and
// L2 steps, run by one wavefront: the Golub-Reinsch SVD of MPI_REAL/tools.c
// (tools.c:113-352) and x = V diag(1/w) V^T b (tools.c:52-105).  U is never
// formed: the reference replaces it by V (tools.c:324-329) and no U-only step
// feeds w, the superdiagonal or V.
//
// The operation sequence is the reference's (bit-identical results).  Loops
// whose iterations are independent are spread over the lanes: lane = column
// (left reflector, right-transform accumulation, the final products) or row
// (right reflector; the QR phase, where each V row is rotated on its own).
//
// What bounds it: a serial chain of FP64 divisions, square roots and ordered
// sums in one wavefront (an inner QR step is 1000 clocks of them).  So the
// rest is kept off that chain: the loops over columns and rotations are not
// unrolled (a kernel unrolled over its templates ran 40 kB of code once per
// solve), w and rv1 live one element per lane and are broadcast by readlane,
// and a reflector's vector is exchanged through LDS, 16 bytes a lane at one
// address, so that every lane holds all of it.  Its sums run over all M
// places with zeros outside its range: that leaves every partial sum as it is
// (they start at +0, so none is -0) and saves a branch per term.  With
// the launch n = 7 takes 34 us and n = 14 96 us (the unrolled form 44 and 127).
#pragma once

#include "aar_common.h"
#include "aar_device.h"
#include "aar_kernels.h"

namespace aar {

// LDS of one solve; the odd pitch keeps row-wise lanes off each other's banks
template <int M> struct LsLds {
    double A[M][M + 1];
    double V[M][M + 1];
    alignas(16) double c0[M];      // a vector every lane is to hold
    alignas(16) double c1[M];
};

// lane l's value, for every lane (l uniform)
__device__ __forceinline__ double ls_bcast(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// a condition every lane agrees on, as a scalar
__device__ __forceinline__ bool ls_all(bool c) { return __builtin_amdgcn_readfirstlane((int)c) != 0; }
// orders one lane's LDS writes before another's reads (one wavefront)
__device__ __forceinline__ void ls_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// all M elements of the vector whose element `lane` this lane holds
template <int M>
__device__ __forceinline__ void ls_all_of(double (&buf)[M], double mine, double (&v)[M])
{
    const int lane = threadIdx.x & 63;
    if (lane < M) buf[lane] = mine;
    ls_sync();
#pragma unroll
    for (int k = 0; k < M; k++) v[k] = buf[k];
    ls_sync();
}

__device__ __forceinline__ double d_pythag(double a, double b)
{
    const double absa = fabs(a), absb = fabs(b);
    const bool g = absa > absb;
    const double hi = g ? absa : absb, lo = g ? absb : absa;
    const double r = hi * sqrt(1.0 + lo * lo / (hi * hi));
    return !g && absb == 0.0 ? 0.0 : r;
}
__device__ __forceinline__ double d_sign(double mag, double s) { return s >= 0.0 ? fabs(mag) : -fabs(mag); }

// Solves the n x n system (n <= M) in L.A (A[i][j]) with the right-hand side
// bv (lane j holds b[j]) by one wavefront; results to ctrl (s, w, V, status,
// done).  flags: LS_TEXTBOOK (the complex solver, no MPI_REAL counterpart)
// runs the left reflector over columns i+1..n-1 only; tools.c:137 also runs it
// over columns 1 <= j < i and j = i, column i itself updated before the
// columns j > i read it, and on some embedded Hermitian systems that order
// does not converge.  LS_GELSD: dgelsd's cutoff.
template <int M>
__device__ __forceinline__ void ls_solve(LsLds<M> &L, const double bv, Ctrl *c, const int n, const int flags)
{
    const int lane = threadIdx.x & 63;
    const int ln = lane < M ? lane : M - 1;            // LDS index of idle lanes
    const bool act = lane < n;
    double wv = 0.0, rv = 0.0;                         // w[lane], rv1[lane]
    double g = 0.0, scale = 0.0, anorm = 0.0, s = 0.0, f = 0.0, h = 0.0;

#pragma unroll
    for (int k = 0; k < M; k++)
        if (act) L.V[k][ln] = 0.0;
    ls_sync();

    // Householder bidiagonalisation (tools.c:122-176)
#pragma unroll 1
    for (int i = 0; i < n; i++) {
        const int l = i + 1;
        rv = lane == i ? scale * g : rv;
        g = s = scale = 0.0;
        const bool low = lane >= i && act;
        double ci = low ? L.A[ln][i] : 0.0;            // A[lane][i], 0 above the diagonal
        double v[M];
        ls_all_of<M>(L.c0, ci, v);
#pragma unroll
        for (int k = 0; k < M; k++) scale += fabs(v[k]);
        if (ls_all(scale != 0.0)) {
            double a[M];                               // this lane's column
#pragma unroll
            for (int k = 0; k < M; k++) a[k] = L.A[k][ln];
            if (low) ci /= scale;
            ls_all_of<M>(L.c0, ci, v);
#pragma unroll
            for (int k = 0; k < M; k++) s += v[k] * v[k];
            f = ls_bcast(ci, i);
            g = -d_sign(sqrt(s), f);
            h = f * g - s;
            f = f - g;
            if (lane == i) ci = f;
#pragma unroll
            for (int k = 0; k < M; k++) v[k] = k == i ? f : v[k];
            // columns j = 1 .. n-1 in the order the sequential loop sees
            // column i: j < i, then j = i, then j > i
            const bool text = flags & LS_TEXTBOOK;
            if (!text && i >= 1) {
                double t = 0.0;
#pragma unroll
                for (int k = 0; k < M; k++) t += v[k] * v[k];
                const double fac = t / h;
                if (low) ci += fac * ci;
                if (lane > i) {                        // those columns see the updated one
#pragma unroll
                    for (int k = 0; k < M; k++) v[k] += fac * v[k];
                }
            }
            double t = 0.0;
#pragma unroll
            for (int k = 0; k < M; k++) t += v[k] * (k >= i && k < n ? a[k] : 0.0);
            const double fac = t / h;
            if (act && (lane > i || (!text && lane >= 1 && lane < i))) {
#pragma unroll
                for (int k = 0; k < M; k++) L.A[k][ln] = k >= i && k < n ? a[k] + fac * v[k] : a[k];
            }
            if (low) {
                ci *= scale;
                L.A[ln][i] = ci;
            }
            ls_sync();
        }
        wv = lane == i ? scale * g : wv;
        g = s = scale = 0.0;
        if (i != n - 1) {
            const bool right = lane >= l && act;
            double ri = right ? L.A[i][ln] : 0.0;      // A[i][lane], 0 up to the diagonal
            ls_all_of<M>(L.c0, ri, v);
#pragma unroll
            for (int k = 0; k < M; k++) scale += fabs(v[k]);
            if (ls_all(scale != 0.0)) {
                double a[M];                           // this lane's row
#pragma unroll
                for (int k = 0; k < M; k++) a[k] = L.A[ln][k];
                if (right) ri /= scale;
                ls_all_of<M>(L.c0, ri, v);
#pragma unroll
                for (int k = 0; k < M; k++) s += v[k] * v[k];
                f = ls_bcast(ri, l);
                g = -d_sign(sqrt(s), f);
                h = f * g - s;
                f = f - g;
                if (lane == l) ri = f;
#pragma unroll
                for (int k = 0; k < M; k++) v[k] = k == l ? f : v[k];
                double t = 0.0;
#pragma unroll
                for (int k = 0; k < M; k++) t += (k >= l && k < n ? a[k] : 0.0) * v[k];
                if (right) rv = ri / h;                // rv1[k] = a[i][k] / h
                ls_all_of<M>(L.c1, rv, v);
                if (right) {
#pragma unroll
                    for (int k = 0; k < M; k++) L.A[ln][k] = k >= l && k < n ? a[k] + t * v[k] : a[k];
                    ri *= scale;
                    L.A[i][ln] = ri;
                }
                ls_sync();
            }
        }
        {
            const double t = fabs(ls_bcast(wv, i)) + fabs(ls_bcast(rv, i));
            anorm = anorm > t ? anorm : t;             // tools.h:21 max()
        }
    }

    // accumulation of right-hand transforms (tools.c:178-196)
#pragma unroll 1
    for (int i = n - 1; i >= 0; i--) {
        const int l = i + 1;
        if (i < n - 1) {
            const double gg = ls_bcast(rv, l);
            const bool right = lane >= l && act;
            if (ls_all(gg != 0.0)) {
                const double ai = right ? L.A[i][ln] : 0.0;
                double a[M], v[M], t = 0.0;
#pragma unroll
                for (int k = 0; k < M; k++) a[k] = L.V[k][ln];
                ls_all_of<M>(L.c0, ai, v);
#pragma unroll
                for (int k = 0; k < M; k++) t += v[k] * (k >= l && k < n ? a[k] : 0.0);
                const double vi = (ai / ls_bcast(ai, l)) / gg;     // v[lane][i]
                ls_all_of<M>(L.c1, vi, v);
                if (right) {
#pragma unroll
                    for (int k = 0; k < M; k++) L.V[k][ln] = k >= l && k < n ? a[k] + t * v[k] : a[k];
                }
            }
            if (right) {
                L.V[i][ln] = 0.0;
                L.V[ln][i] = 0.0;
            }
        }
        if (lane == i) L.V[i][ln] = 1.0;
        ls_sync();
    }

    // implicit-shift QR on the bidiagonal (tools.c:254-350): lane = V row
    int status = 0;
    double *vrow = L.V[ln];
#pragma unroll 1
    for (int k = n - 1; k >= 0 && !status; k--) {
#pragma unroll 1
        for (int its = 0; its <= 250; its++) {
            // the largest ll <= k where rv1[ll] is negligible (flag = 0), or
            // w[ll-1] is (flag = 1)
            const double wprev = __shfl_up(wv, 1, 64);
            const bool c1 = lane <= k && (double)(fabs(rv) + anorm) == anorm;
            const bool c2 = lane >= 1 && lane <= k && (double)(fabs(wprev) + anorm) == anorm;
            const unsigned long long m1 = __ballot(c1), m2 = __ballot(c2);
            const unsigned long long mm = m1 | m2;
            const int l = mm ? 63 - __clzll((long long)mm) : 0;
            const bool flag = mm ? !((m1 >> l) & 1ull) : true;
            if (flag) {
                double cc = 0.0;
                s = 1.0;
#pragma unroll 1
                for (int i = l; i <= k; i++) {
                    const double r = ls_bcast(rv, i);
                    f = s * r;
                    rv = lane == i ? cc * r : rv;
                    if (ls_all((double)(fabs(f) + anorm) == anorm)) break;
                    g = ls_bcast(wv, i);
                    h = d_pythag(f, g);
                    wv = lane == i ? h : wv;
                    h = 1.0 / h;
                    cc = g * h;
                    s = -f * h;
                }
            }
            double z = ls_bcast(wv, k);
            if (l == k) {
                if (ls_all(z < 0.0)) {
                    wv = lane == k ? -z : wv;
                    if (act) vrow[k] = -vrow[k];
                }
                break;
            }
            if (its == 250) {
                status = 1;
                break;
            }
            double x = ls_bcast(wv, l);
            const int nm = k - 1;
            double y = ls_bcast(wv, nm);
            g = ls_bcast(rv, nm);
            h = ls_bcast(rv, k);
            f = ((y - z) * (y + z) + (g - h) * (g + h)) / (2.0 * h * y);
            g = d_pythag(f, 1.0);
            f = ((x - z) * (x + z) + h * ((y / (f + d_sign(g, f))) - h)) / x;
            double cc = 1.0;
            s = 1.0;
            double vx = vrow[l];
#pragma unroll 1
            for (int j = l; j < k; j++) {
                const int i = j + 1;
                const double vz = vrow[i];
                g = ls_bcast(rv, i);
                y = ls_bcast(wv, i);
                h = s * g;
                g = cc * g;
                z = d_pythag(f, h);
                rv = lane == j ? z : rv;
                cc = f / z;
                s = h / z;
                f = x * cc + g * s;
                g = g * cc - x * s;
                h = y * s;
                y *= cc;
                if (act) vrow[j] = vx * cc + vz * s;
                vx = vz * cc - vx * s;
                z = d_pythag(f, h);
                wv = lane == j ? z : wv;
                if (ls_all(z != 0.0)) {
                    z = 1.0 / z;
                    cc = f * z;
                    s = h * z;
                }
                f = cc * g + s * y;
                x = cc * y - s * g;
            }
            if (act) vrow[k] = vx;
            rv = lane == l ? 0.0 : rv;
            rv = lane == k ? f : rv;
            wv = lane == k ? x : wv;
        }
    }
    ls_sync();

    // truncation (tools.c:331-335: w < n w_max 2.22044605e-16; with
    // LS_GELSD, LAPACK dgelsd's rcond = -1 rule of the PETSc variant:
    // w <= 2^-53 w_max) and x = V diag(1/w) V^T b (tools.c:76-94)
    double wmax = 0.0;
#pragma unroll 1
    for (int j = 0; j < n; j++) {
        const double t = ls_bcast(wv, j);
        wmax = t > wmax ? t : wmax;
    }
    if (flags & LS_GELSD) {
        if (wv <= 1.1102230246251565e-16 * wmax) wv = 0.0;
    } else {
        if (wv < n * wmax * (2.22044605e-16)) wv = 0.0;
    }
    double t = 0.0;
#pragma unroll 4
    for (int i = 0; i < n; i++) t += L.V[i][ln] * ls_bcast(bv, i);
    const double tl = act && wv != 0.0 ? t / wv : 0.0;
    t = 0.0;
#pragma unroll 4
    for (int j = 0; j < n; j++) t += vrow[j] * ls_bcast(tl, j);
    if (act) {
        c->s[lane] = t;
        c->w[lane] = wv;
    }
    for (int e = lane; e < n * n; e += 64) c->V[e] = L.V[e / n][e % n];
    if (status && lane == 0) {
        // tools.c:270 exits the process; here the solve stops with a status
        c->status = 1;
        c->done = 1;
    }
}

// the system of ctrl->G: FtF[i][j] = allredvec[j*m + i], Ftf[j] =
// allredvec[m*m + j] (AAR.c:214-221)
template <int M>
__device__ __forceinline__ void ls_from_ctrl(LsLds<M> &L, Ctrl *c, const int n, const int flags)
{
    const int lane = threadIdx.x & 63;
    for (int e = lane; e < n * n; e += 64) L.A[e % n][e / n] = c->G[e];
    const double bv = lane < n ? c->G[n * n + lane] : 0.0;
    ls_sync();
    ls_solve<M>(L, bv, c, n, flags);
}

}  // namespace aar
