// ls.hip -- the m x m least-squares solve of the Anderson, Galerkin and L2
// steps on the device (one wavefront).
#include "aar_common.h"
#include "aar_device.h"
#include "aar_kernels.h"

namespace aar {

// ---------------------------------------------------------------------------
// m x m pseudo-inverse solve: the Golub-Reinsch SVD of MPI_REAL/tools.c
// (tools.c:113-352) and x = V diag(1/w) V^T b (tools.c:52-105).  U is
// never formed: the reference replaces it by V (tools.c:324-329) and no
// U-only step feeds w, the superdiagonal or V.
// ---------------------------------------------------------------------------
__device__ __attribute__((always_inline)) inline double d_pythag(double a, double b)
{
    const double absa = fabs(a), absb = fabs(b);
    if (absa > absb) return absa * sqrt(1.0 + absb * absb / (absa * absa));
    return absb == 0.0 ? 0.0 : absb * sqrt(1.0 + absa * absa / (absb * absb));
}
__device__ inline double d_sign(double mag, double s) { return s >= 0.0 ? fabs(mag) : -fabs(mag); }

// ---------------------------------------------------------------------------
// The pinv is executed by one wavefront.  The operation sequence is the
// reference's (bit-identical results); loops whose iterations are
// independent are spread over the lanes -- lane = column (left reflector,
// right-transform accumulation, the final products) or row (right
// reflector; the QR phase, where each V row is rotated on its own and
// stays in the lane's registers).  Scalars (w, rv1, the reflector and
// rotation coefficients) are computed by every lane alike.  The left
// reflector of tools.c:137 also runs over columns j < i and j = i; column
// i itself is updated before the columns j > i read it, as in the
// sequential loop.  textbook = 1 (the complex solver, no MPI_REAL
// counterpart) runs the textbook step over columns i+1..n-1 only: on some
// embedded Hermitian systems the tools.c order does not converge.
// ---------------------------------------------------------------------------
template <int M, int k>
__device__ __attribute__((always_inline)) inline void wgr_qr_step(double (&w)[M], double (&rv1)[M], double (&vr)[M],
                                                                   const double anorm, const int n, int &status)
{
    double g = 0.0, s = 0.0, f = 0.0, h = 0.0;
    if (k < n && !status) {
        for (int its = 0; its <= 250; its++) {
            int flag = 1, l = 0;
            bool found = false;
#pragma unroll
            for (int ll = k; ll >= 0; ll--) {
                if (!found) {
                    if ((double)(fabs(rv1[ll]) + anorm) == anorm) {
                        flag = 0;
                        l = ll;
                        found = true;
                    } else if (ll >= 1 && (double)(fabs(w[ll >= 1 ? ll - 1 : 0]) + anorm) == anorm) {
                        l = ll;
                        found = true;
                    }
                }
            }
            if (flag) {
                double c = 0.0;
                s = 1.0;
                bool stop = false;
#pragma unroll
                for (int i = 0; i <= k; i++) {
                    if (i >= l && !stop) {
                        f = s * rv1[i];
                        rv1[i] = c * rv1[i];
                        if ((double)(fabs(f) + anorm) == anorm) {
                            stop = true;
                        } else {
                            g = w[i];
                            h = d_pythag(f, g);
                            w[i] = h;
                            h = 1.0 / h;
                            c = g * h;
                            s = -f * h;
                        }
                    }
                }
            }
            double z = w[k];
            if (l == k) {
                if (z < 0.0) {
                    w[k] = -z;
                    vr[k] = -vr[k];
                }
                break;
            }
            if (its == 250) {
                status = 1;
                break;
            }
            double x = 0.0;
#pragma unroll
            for (int ll = 0; ll <= k; ll++)
                if (ll == l) x = w[ll];
            const int nm = k - 1;
            double y = w[nm >= 0 ? nm : 0];
            g = rv1[nm >= 0 ? nm : 0];
            h = rv1[k];
            f = ((y - z) * (y + z) + (g - h) * (g + h)) / (2.0 * h * y);
            g = d_pythag(f, 1.0);
            f = ((x - z) * (x + z) + h * ((y / (f + d_sign(g, f))) - h)) / x;
            double c = 1.0;
            s = 1.0;
#pragma unroll
            for (int j = 0; j < k; j++) {
                if (j >= l) {
                    const int i = j + 1;
                    g = rv1[i];
                    y = w[i];
                    h = s * g;
                    g = c * g;
                    z = d_pythag(f, h);
                    rv1[j] = z;
                    c = f / z;
                    s = h / z;
                    f = x * c + g * s;
                    g = g * c - x * s;
                    h = y * s;
                    y *= c;
                    {
                        const double vx = vr[j], vz = vr[i];
                        vr[j] = vx * c + vz * s;
                        vr[i] = vz * c - vx * s;
                    }
                    z = d_pythag(f, h);
                    w[j] = z;
                    if (z != 0.0) {
                        z = 1.0 / z;
                        c = f * z;
                        s = h * z;
                    }
                    f = c * g + s * y;
                    x = c * y - s * g;
                }
            }
#pragma unroll
            for (int ll = 0; ll <= k; ll++)
                if (ll == l) rv1[ll] = 0.0;
            rv1[k] = f;
            w[k] = x;
        }
    }
}

template <int M, int k>
struct WGrQr {
    __device__ __attribute__((always_inline)) static inline void run(double (&w)[M], double (&rv1)[M], double (&vr)[M],
                                                                      const double anorm, const int n, int &status)
    {
        wgr_qr_step<M, k>(w, rv1, vr, anorm, n, status);
        WGrQr<M, k - 1>::run(w, rv1, vr, anorm, n, status);
    }
};
template <int M>
struct WGrQr<M, -1> {
    __device__ static inline void run(double (&)[M], double (&)[M], double (&)[M], const double, const int, int &) {}
};

template <int M>
__device__ __forceinline__ void ls_body(Ctrl *c, const int n, const int flags)
{
    __shared__ double A[M][M];
    __shared__ double V[M][M];
    __shared__ double T[M];
    if (c->done) return;
    const int lane = threadIdx.x;
    // FtF[i][j] = allredvec[j*m + i], Ftf[j] = allredvec[m*m + j] (AAR.c:214-221)
    for (int e = lane; e < M * M; e += 64) {
        const int i = e / M, j = e % M;
        A[i][j] = (i < n && j < n) ? c->G[j * n + i] : 0.0;
        V[i][j] = 0.0;
    }
    __syncthreads();

    double w[M], rv1[M];
#pragma unroll
    for (int i = 0; i < M; i++) {
        w[i] = 0.0;
        rv1[i] = 0.0;
    }
    double g = 0.0, scale = 0.0, anorm = 0.0, s = 0.0, f = 0.0, h = 0.0;

    // Householder bidiagonalisation (tools.c:122-176)
#pragma unroll
    for (int i = 0; i < M; i++) {
        if (i < n) {
            const int l = i + 1;
            rv1[i] = scale * g;
            g = s = scale = 0.0;
            for (int k = i; k < n; k++) scale += fabs(A[k][i]);
            if (scale != 0.0) {
                __syncthreads();
                if (lane >= i && lane < n) A[lane][i] /= scale;
                __syncthreads();
                for (int k = i; k < n; k++) s += A[k][i] * A[k][i];
                f = A[i][i];
                g = -d_sign(sqrt(s), f);
                h = f * g - s;
                __syncthreads();
                if (lane == 0) A[i][i] = f - g;
                __syncthreads();
                // columns j = 1 .. n-1 in the order the sequential loop sees
                // column i: j < i, then j = i, then j > i
                auto colupd = [&](int j) {
                    double t = 0.0;
                    for (int k = i; k < n; k++) t += A[k][i] * A[k][j];
                    const double fac = t / h;
                    for (int k = i; k < n; k++) A[k][j] += fac * A[k][i];
                };
                if (!(flags & LS_TEXTBOOK)) {
                    if (lane >= 1 && lane < i && lane < n) colupd(lane);
                    __syncthreads();
                    if (i >= 1 && lane == i) colupd(i);
                    __syncthreads();
                }
                if (lane > i && lane >= 1 && lane < n) colupd(lane);
                __syncthreads();
                if (lane >= i && lane < n) A[lane][i] *= scale;
                __syncthreads();
            }
            w[i] = scale * g;
            g = s = scale = 0.0;
            if (i != n - 1) {
                for (int k = l; k < n; k++) scale += fabs(A[i][k]);
                if (scale != 0.0) {
                    __syncthreads();
                    if (lane >= l && lane < n) A[i][lane] /= scale;
                    __syncthreads();
                    for (int k = l; k < n; k++) s += A[i][k] * A[i][k];
                    f = A[i][l < M ? l : M - 1];
                    g = -d_sign(sqrt(s), f);
                    h = f * g - s;
                    __syncthreads();
                    if (lane == 0) A[i][l < M ? l : M - 1] = f - g;
                    __syncthreads();
                    // rv1[k] = a[i][k] / h, kept by every lane
#pragma unroll
                    for (int k = 0; k < M; k++)
                        if (k >= l && k < n) rv1[k] = A[i][k] / h;
                    if (lane >= l && lane < n) {
                        double t = 0.0;
                        for (int k = l; k < n; k++) t += A[lane][k] * A[i][k];
#pragma unroll
                        for (int k = 0; k < M; k++)
                            if (k >= l && k < n) A[lane][k] += t * rv1[k];
                    }
                    __syncthreads();
                    if (lane >= l && lane < n) A[i][lane] *= scale;
                    __syncthreads();
                }
            }
            {
                const double t = fabs(w[i]) + fabs(rv1[i]);
                anorm = anorm > t ? anorm : t;       // tools.h:21 max()
            }
        }
    }

    // accumulation of right-hand transforms (tools.c:178-196)
#pragma unroll
    for (int i = M - 1; i >= 0; i--) {
        if (i < n) {
            if (i < n - 1) {
                const int l = i + 1;
                const double gg = rv1[l < M ? l : M - 1];
                if (gg != 0.0) {
                    const double ail = A[i][l < M ? l : M - 1];
                    if (lane >= l && lane < n) V[lane][i] = (A[i][lane] / ail) / gg;
                    __syncthreads();
                    if (lane >= l && lane < n) {
                        double t = 0.0;
                        for (int k = l; k < n; k++) t += A[i][k] * V[k][lane];
                        for (int k = l; k < n; k++) V[k][lane] += t * V[k][i];
                    }
                    __syncthreads();
                }
                if (lane >= l && lane < n) {
                    V[i][lane] = 0.0;
                    V[lane][i] = 0.0;
                }
                __syncthreads();
            }
            if (lane == 0) V[i][i] = 1.0;
            __syncthreads();
        }
    }

    // implicit-shift QR on the bidiagonal (tools.c:254-350): lane = V row
    double vr[M];
#pragma unroll
    for (int j = 0; j < M; j++) vr[j] = (lane < n) ? V[lane < M ? lane : 0][j] : 0.0;
    int status = 0;
    WGrQr<M, M - 1>::run(w, rv1, vr, anorm, n, status);
    __syncthreads();
    if (lane < n) {
#pragma unroll
        for (int j = 0; j < M; j++) V[lane][j] = vr[j];
    }
    __syncthreads();

    // truncation (tools.c:331-335: w < n w_max 2.22044605e-16; with
    // LS_GELSD, LAPACK dgelsd's rcond = -1 rule of the PETSc variant:
    // w <= 2^-53 w_max) and x = V diag(1/w) V^T b (tools.c:76-94)
    double wmax = 0.0;
#pragma unroll
    for (int j = 0; j < M; j++)
        if (j < n && w[j] > wmax) wmax = w[j];
    if (flags & LS_GELSD) {
        const double tol = 1.1102230246251565e-16 * wmax;
#pragma unroll
        for (int j = 0; j < M; j++)
            if (j < n && w[j] <= tol) w[j] = 0.0;
    } else {
        const double wmin = n * wmax * (2.22044605e-16);
#pragma unroll
        for (int j = 0; j < M; j++)
            if (j < n && w[j] < wmin) w[j] = 0.0;
    }
    if (lane < n) {
        double wl = 0.0;
#pragma unroll
        for (int j = 0; j < M; j++)
            if (j == lane) wl = w[j];
        double t = 0.0;
        if (wl != 0.0) {
            for (int i = 0; i < n; i++) t += V[i][lane] * c->G[n * n + i];
            t /= wl;
        }
        T[lane] = t;
    }
    __syncthreads();
    if (lane < n) {
        double t = 0.0;
        for (int jj = 0; jj < n; jj++) t += V[lane][jj] * T[jj];
        c->s[lane] = t;
        double wl = 0.0;
#pragma unroll
        for (int j = 0; j < M; j++)
            if (j == lane) wl = w[j];
        c->w[lane] = wl;
        for (int q = 0; q < n; q++) c->V[lane * n + q] = V[lane][q];
    }
    if (status && lane == 0) {
        // tools.c:270 exits the process; here the solve stops with a status
        c->status = 1;
        c->done = 1;
    }
}

template <int M>
__global__ __launch_bounds__(64) void ls_kernel(Ctrl *c, int n, int flags)
{
    ls_body<M>(c, n, flags);
}

// one wavefront per solve of a batch
template <int M>
__global__ __launch_bounds__(64) void ls_batch_kernel(Ctrl *const *ctrls, int n)
{
    ls_body<M>(ctrls[blockIdx.x], n, 0);
}

hipError_t launch_ls_batch(Ctrl *const *ctrls, int count, int n, hipStream_t st)
{
    if (n < 1 || n > MAXM_LS || count < 1) return hipErrorInvalidValue;
    if (n > MAXM_BATCH) return hipErrorInvalidValue;
    if (n <= 8) hipLaunchKernelGGL((ls_batch_kernel<8>), dim3(count), dim3(64), 0, st, ctrls, n);
    else hipLaunchKernelGGL((ls_batch_kernel<16>), dim3(count), dim3(64), 0, st, ctrls, n);
    return hipGetLastError();
}

hipError_t launch_ls(Ctrl *ctrl, int n, int flags, hipStream_t st)
{
    if (n < 1 || n > MAXM_LS) return hipErrorInvalidValue;
    if (n <= 8) hipLaunchKernelGGL((ls_kernel<8>), dim3(1), dim3(64), 0, st, ctrl, n, flags);
    else if (n <= 16) hipLaunchKernelGGL((ls_kernel<16>), dim3(1), dim3(64), 0, st, ctrl, n, flags);
    else hipLaunchKernelGGL((ls_kernel<32>), dim3(1), dim3(64), 0, st, ctrl, n, flags);
    return hipGetLastError();
}

}  // namespace aar
