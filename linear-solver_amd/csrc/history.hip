// history.hip -- Anderson / Galerkin / L2 history kernels of libaar_hip.
//
// The reference builds its normal equations with m(m+1)/2 + m (AAR, PL2R)
// or m^2 + m (PGR) separate N-length dot passes over stored difference
// columns (MPI_REAL/AAR.c:192-210, PGR.c:188-204, PL2R.c:187-204) and then
// re-reads 2m columns for the update (AAR.c:225-231, PGR.c:117-121).
// Here the iterates x_k and residuals f_k themselves live in ring buffers
// of m+1 slots, difference columns are formed on the fly with the same
// subtraction the reference stores (DX = x - x_old, DF = f - f_old), and
// the whole normal-equation build is ONE pass over the m+1 slots with all
// products accumulated in FP64 registers.  The m x m solve runs on device.
#include <type_traits>

#include "history.h"
#include "ls_body.h"

namespace aar {

// The system built from the sums of a Gram (AAR.c:192-212, PGR.c:188-206):
// reference allredvec layout, [j*m + i] = col_i . col_j, [m*m + j] = col_j . f;
// missing columns are zero.  Every thread of the block writes its entries.
// mm: the columns the sums were made for (products (j, q) at j*mm + q for
// kind 1, else the lower triangle by rows; then the right-hand sides).
struct GramFin {
    int m, mm, kind, nvalid, it, direct;
    int nblocks;
    const double *partials;
    Ctrl *ctrl;
};
__device__ __forceinline__ int gram_values(const GramFin &a)
{
    return (a.kind == 1 ? a.mm * a.mm : a.mm * (a.mm + 1) / 2) + a.mm;
}
// value e < m*m + m of the layout
__device__ __forceinline__ double gram_entry(const GramFin &a, const double *sums, int e)
{
    const int m = a.m, nv = a.nvalid;
    // age of the reference's column c (ref_col inverted)
    auto age = [&](int c) { return a.direct ? c : ((a.it - 2 - c) % m + m) % m; };
    if (e >= m * m) {
        const int k = age(e - m * m);
        return k < nv ? sums[gram_values(a) - a.mm + k] : 0.0;
    }
    const int j = age(e / m), q = age(e % m);
    if (j >= nv || q >= nv) return 0.0;
    if (a.kind == 1) return sums[j * a.mm + q];
    return j > q ? sums[j * (j + 1) / 2 + q] : sums[q * (q + 1) / 2 + j];
}

template <typename T, int MM, int KIND>
__device__ inline void gram_layout(const GramArgs<T> &a, const double *sums)
{
    const GramFin f = {a.m, MM, KIND, a.nvalid, a.it, a.direct, a.nblocks, a.partials, a.ctrl};
    for (int e = threadIdx.x; e < a.m * a.m + a.m; e += blockDim.x) a.ctrl->G[e] = gram_entry(f, sums, e);
}

// ---------------------------------------------------------------------------
// normal equations, one pass over the m+1 ring slots
// ---------------------------------------------------------------------------
template <typename T, int MM, int KIND>
__global__ __launch_bounds__(BLOCK) void gram_kernel(const GramArgs<T> a)
{
    constexpr int NG = (KIND == 1) ? MM * MM : MM * (MM + 1) / 2;
    constexpr int NA = NG + MM;
    static_assert(NA <= GRAM_NA_MAX, "partials buffers hold GRAM_NA_MAX per block");
    constexpr int NS = MM + 1;
    __shared__ double scratch[NA * (BLOCK / 64)];
    __shared__ double sums[NA];
    if (a.ctrl->done) return;

    const int m = a.m, nv = a.nvalid, dir = a.direct;
    const T *D = (KIND == 0) ? a.F : a.Y;     // ring of the DF columns
    const T *pd[NS], *px[NS];
    bool use[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        use[k] = dir ? (k < nv) : (k <= nv);
        const size_t off = (size_t)(use[k] ? a.slot[k] : 0) * a.ld;
        pd[k] = D + off;
        px[k] = a.F + off;
    }
    const T *pf = (KIND == 0 ? a.F : a.Y) + (size_t)a.fslot * a.ld;

    double acc[NA];
#pragma unroll
    for (int k = 0; k < NA; k++) acc[k] = 0.0;

    // one point: DF (and DX) columns by age, then all products in FP64
    auto point = [&](T fv, const T (&vd)[NS], const T (&vx)[NS]) {
        double d[MM], e[MM];
#pragma unroll
        for (int k = 0; k < MM; k++) {
            d[k] = 0.0;
            e[k] = 0.0;
            if (k < nv) {
                d[k] = dir ? (double)vd[k] : (double)(vd[k] - vd[k + 1]);   // DF = f - f_old
                if constexpr (KIND == 1)
                    e[k] = dir ? (double)vx[k] : (double)(vx[k] - vx[k + 1]);   // DX = x - x_old
            }
        }
        const double fd = (double)fv;
        if constexpr (KIND == 1) {
#pragma unroll
            for (int j = 0; j < MM; j++) {
#pragma unroll
                for (int q = 0; q < MM; q++) acc[j * MM + q] += e[q] * d[j];   // DX_q . DF_j
                acc[NG + j] += e[j] * fd;                                      // DX_j . f
            }
        } else {
            int t = 0;
#pragma unroll
            for (int j = 0; j < MM; j++) {
#pragma unroll
                for (int q = 0; q <= j; q++) acc[t++] += d[q] * d[j];          // DF_q . DF_j
                acc[NG + j] += d[j] * fd;                                      // DF_j . f
            }
        }
    };

    // A fixed point-to-thread assignment, so the reduction order is fixed:
    // block b walks the chunks b, b + nblocks, ... of CHUNK_V 16-byte
    // vectors, each contiguous (measured 13% faster at 512^3 than a grid
    // stride of one vector per thread: every CU streams contiguous memory).
    // VW consecutive points per 16-byte load when N is a multiple of VW
    // (every ring slot is 256-byte aligned).  The newest slot is both the
    // age-0 column end and f (the residual ring of AAR; the A x ring of
    // PGR/PL2R, f = b - A x): one load.
    constexpr int VW = 16 / sizeof(T);
    using VT = T __attribute__((ext_vector_type(VW)));
    const bool f_is_d0 = !dir && a.fslot == a.slot[0];
    const long n = a.n;
    const long stride = (long)gridDim.x * BLOCK;
    const bool vec_ok = (n % VW) == 0 && (KIND == 0 || ((uintptr_t)a.b % 16) == 0);
    if (vec_ok) {
        const long nq = n / VW;
        for (long iq = chunk_first(a.chunk); iq < nq; iq = chunk_next(iq, a.chunk)) {
            const long i = VW * iq;
            VT vd[NS], vx[NS];
#pragma unroll
            for (int k = 0; k < NS; k++) {
                vd[k] = (VT)(T)0;
                vx[k] = (VT)(T)0;
                if (use[k]) {
                    // streamed once per launch: not kept in the caches (2-8%
                    // faster at 512^3 than cached loads)
                    vd[k] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(pd[k] + i));
                    if constexpr (KIND == 1) vx[k] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(px[k] + i));
                }
            }
            VT fv = f_is_d0 ? vd[0] : *reinterpret_cast<const VT *>(pf + i);
            if constexpr (KIND != 0) fv = *reinterpret_cast<const VT *>(a.b + i) - fv;   // PGR.c:102-103
#pragma unroll
            for (int e = 0; e < VW; e++) {
                T sd[NS], sx[NS];
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    sd[k] = vd[k][e];
                    sx[k] = vx[k][e];
                }
                point(fv[e], sd, sx);
            }
        }
    } else {
        for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) {
            T vd[NS], vx[NS];
#pragma unroll
            for (int k = 0; k < NS; k++) {
                vd[k] = use[k] ? pd[k][i] : (T)0;
                vx[k] = (KIND == 1 && use[k]) ? px[k][i] : (T)0;
            }
            T f = pf[i];
            if constexpr (KIND != 0) f = a.b[i] - f;
            point(f, vd, vx);
        }
    }

    // value-major partials: each value's per-block sums are contiguous
    block_reduce_to_vm<NA>(acc, a.partials + blockIdx.x, a.nblocks, scratch);
    if (!a.counter) return;                     // two-pass: gram_finish_kernel follows
    if (last_block_arrive(a.counter, gridDim.x)) {
        final_sum_vm(a.partials, a.nblocks, NA, sums);
        gram_layout<T, MM, KIND>(a, sums);
        if (threadIdx.x == 0) *a.counter = 0u;
    }
}

// Second pass of the normal-equation build, and the m x m solve: one block
// sums the per-block partials in a fixed order (one wavefront per value,
// contiguous reads), every thread lays out its entries, and the first
// wavefront solves (ls_body.h).  One launch instead of two, and sixteen
// wavefronts on the sums instead of four: at m = 7 on 512 blocks the finish
// (17 us, half of it one thread's layout) and the solve (63 us) took 80 us a
// cycle at 512^3, now 45.  Larger systems leave a wavefront more registers.
template <int M> constexpr int GFIN_NT = M <= 8 ? 1024 : (M <= 16 ? 512 : 256);

template <int M>
__global__ __launch_bounds__(GFIN_NT<M>) void gram_finish_kernel(const GramFin a, int flags)
{
    __shared__ double sums[M * M + M];
    __shared__ LsLds<M> L;
    Ctrl *c = a.ctrl;
    if (c->done) return;
    final_sum_vm<GFIN_NT<M>>(a.partials, a.nblocks, gram_values(a), sums);
    const int m = a.m;
    for (int e = threadIdx.x; e < m * m + m; e += GFIN_NT<M>) {
        const double v = gram_entry(a, sums, e);
        c->G[e] = v;
        // FtF[i][j] = allredvec[j*m + i] (AAR.c:214-221)
        if (e < m * m) L.A[e % m][e / m] = v;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x;
    ls_solve<M>(L, lane < m ? gram_entry(a, sums, m * m + lane) : 0.0, c, m, flags);
}

// columns of the instantiation that a history of m runs: the reference's
// default m = 7 (AAR) has its own, 35 accumulators and 8 loads per point
// instead of MAXM_FAST's 44 and 9; the READMEs' m = 13 too
static int gram_columns(int kind, int m)
{
    if (kind == 0 && m == 7) return 7;
    return m <= MAXM_FAST ? MAXM_FAST : (m == 13 ? 13 : (m <= MAXM_MID ? MAXM_MID : MAXM));
}

template <typename T>
hipError_t launch_gram_solve(const GramArgs<T> &a, int flags, hipStream_t st)
{
    const int mm = gram_columns(a.kind, a.m);
    if (a.counter && a.m <= MAXM_MID) return launch_ls(a.ctrl, a.m, flags, st);    // ctrl->G is there
    const GramFin f = {a.m, mm, a.kind, a.nvalid, a.it, a.direct, a.nblocks, a.partials, a.ctrl};
    const dim3 grid(1);
    if (mm <= 8) hipLaunchKernelGGL((gram_finish_kernel<8>), grid, dim3(GFIN_NT<8>), 0, st, f, flags);
    else if (mm <= 16) hipLaunchKernelGGL((gram_finish_kernel<16>), grid, dim3(GFIN_NT<16>), 0, st, f, flags);
    else hipLaunchKernelGGL((gram_finish_kernel<32>), grid, dim3(GFIN_NT<32>), 0, st, f, flags);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Normal equations beyond m = 16 (560 or 1056 products: more than one pass
// of four wavefronts holds in registers).  The products are cut into NSL
// slices of consecutive products; each of a block's four wavefronts owns one
// slice and walks the block's chunks (the later wavefronts' loads come from
// the caches).  One launch (pass) covers four slices, so HBM reads each
// needed ring slot once per pass, and no accumulator leaves the registers.
// ---------------------------------------------------------------------------
template <int MM, int KIND>
struct GramIdx {
    static constexpr int NG = (KIND == 1) ? MM * MM : MM * (MM + 1) / 2;
    static constexpr int NA = NG + MM;
    // product t: column pair (j, q) of G, or (j, -1) for col_j . f
    static constexpr int j_of(int t)
    {
        if (t >= NG) return t - NG;
        if (KIND == 1) return t / MM;
        int j = 0;
        while ((j + 1) * (j + 2) / 2 <= t) j++;
        return j;
    }
    static constexpr int q_of(int t)
    {
        if (t >= NG) return -1;
        if (KIND == 1) return t % MM;
        const int j = j_of(t);
        return t - j * (j + 1) / 2;
    }
};

template <typename T, int MM, int KIND, int W, int NSL>
__device__ __forceinline__ void gram_split_part(const GramArgs<T> &a)
{
    using Ix = GramIdx<MM, KIND>;
    constexpr int NA = Ix::NA;
    constexpr int PER = (NA + NSL - 1) / NSL;
    constexpr int T0 = W * PER < NA ? W * PER : NA;
    constexpr int T1 = (W + 1) * PER < NA ? (W + 1) * PER : NA;
    if constexpr (T1 <= T0) return;     // a slice past the last product
    constexpr int NT = T1 > T0 ? T1 - T0 : 1;
    constexpr int NS = MM + 1;
    const int m = a.m, nv = a.nvalid, dir = a.direct;
    (void)m;
    const T *D = (KIND == 0) ? a.F : a.Y;
    const T *pd[NS], *px[NS];
    bool use[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        use[k] = dir ? (k < nv) : (k <= nv);
        const size_t off = (size_t)(use[k] ? a.slot[k] : 0) * a.ld;
        pd[k] = D + off;
        px[k] = a.F + off;
    }
    const T *pf = (KIND == 0 ? a.F : a.Y) + (size_t)a.fslot * a.ld;
    const bool f_is_d0 = !dir && a.fslot == a.slot[0];
    double acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = 0.0;

    // this wavefront's products at one point
    auto point = [&](T fv, const T (&vd)[NS], const T (&vx)[NS]) {
        double d[MM], e[MM];
#pragma unroll
        for (int k = 0; k < MM; k++) {
            d[k] = 0.0;
            e[k] = 0.0;
            if (k < nv) {
                d[k] = dir ? (double)vd[k] : (double)(vd[k] - vd[k + 1]);        // DF = f - f_old
                if constexpr (KIND == 1)
                    e[k] = dir ? (double)vx[k] : (double)(vx[k] - vx[k + 1]);    // DX = x - x_old
            }
        }
        const double fd = (double)fv;
#pragma unroll
        for (int t = T0; t < T1; t++) {
            constexpr int dummy = 0;
            (void)dummy;
            const int j = Ix::j_of(t), q = Ix::q_of(t);
            const double u = (q < 0) ? fd : (KIND == 1 ? e[q < 0 ? 0 : q] : d[q < 0 ? 0 : q]);
            const double v = (q < 0 && KIND == 1) ? e[j] : d[j];
            acc[t - T0] += u * v;
        }
    };

    const int lane = threadIdx.x & 63;
    constexpr int VW = 16 / sizeof(T);
    using VT = T __attribute__((ext_vector_type(VW)));
    const long n = a.n;
    const bool vec_ok = (n % VW) == 0 && (KIND == 0 || ((uintptr_t)a.b % 16) == 0);
    const long nq = vec_ok ? n / VW : n;
    for (long c0 = (long)blockIdx.x * CHUNK_V; c0 < nq; c0 += (long)gridDim.x * CHUNK_V) {
        const long c1 = c0 + CHUNK_V < nq ? c0 + CHUNK_V : nq;
        if (vec_ok) {
            for (long iq = c0 + lane; iq < c1; iq += 64) {
                const long i = VW * iq;
                VT vd[NS], vx[NS];
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    vd[k] = (VT)(T)0;
                    vx[k] = (VT)(T)0;
                    if (use[k]) {
                        vd[k] = *reinterpret_cast<const VT *>(pd[k] + i);
                        if constexpr (KIND == 1) vx[k] = *reinterpret_cast<const VT *>(px[k] + i);
                    }
                }
                VT fv = f_is_d0 ? vd[0] : *reinterpret_cast<const VT *>(pf + i);
                if constexpr (KIND != 0) fv = *reinterpret_cast<const VT *>(a.b + i) - fv;   // PGR.c:102-103
#pragma unroll
                for (int e = 0; e < VW; e++) {
                    T sd[NS], sx[NS];
#pragma unroll
                    for (int k = 0; k < NS; k++) {
                        sd[k] = vd[k][e];
                        sx[k] = vx[k][e];
                    }
                    point(fv[e], sd, sx);
                }
            }
        } else {
            for (long i = c0 + lane; i < c1; i += 64) {
                T vd[NS], vx[NS];
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    vd[k] = use[k] ? pd[k][i] : (T)0;
                    vx[k] = (KIND == 1 && use[k]) ? px[k][i] : (T)0;
                }
                T f = pf[i];
                if constexpr (KIND != 0) f = a.b[i] - f;
                point(f, vd, vx);
            }
        }
    }
    // this wavefront owns products T0..T1-1: one value-major partial each
#pragma unroll
    for (int t = T0; t < T1; t++) {
        const double v = wave_sum(acc[t - T0]);
        if (lane == 0) a.partials[(size_t)t * a.nblocks + blockIdx.x] = v;
    }
}

// pass PASS of NPASS: wavefront w owns slice 4 PASS + w of 4 NPASS
template <typename T, int MM, int KIND, int PASS = 0, int NPASS = 1>
__global__ __launch_bounds__(BLOCK) void gram_split_kernel(const GramArgs<T> a)
{
    static_assert(BLOCK == 256, "four wavefronts share the products");
    constexpr int NA = GramIdx<MM, KIND>::NA;
    constexpr int NSL = 4 * NPASS;
    static_assert(NA <= GRAM_NA_MAX, "partials buffers hold GRAM_NA_MAX per block");
    __shared__ double sums[NA];
    if (a.ctrl->done) return;
    switch (threadIdx.x >> 6) {
    case 0: gram_split_part<T, MM, KIND, 4 * PASS + 0, NSL>(a); break;
    case 1: gram_split_part<T, MM, KIND, 4 * PASS + 1, NSL>(a); break;
    case 2: gram_split_part<T, MM, KIND, 4 * PASS + 2, NSL>(a); break;
    default: gram_split_part<T, MM, KIND, 4 * PASS + 3, NSL>(a); break;
    }
    // two-pass (gram_finish_kernel follows), always so for several passes
    if (NPASS > 1 || !a.counter) return;
    if (last_block_arrive(a.counter, gridDim.x)) {
        final_sum_vm(a.partials, a.nblocks, NA, sums);
        gram_layout<T, MM, KIND>(a, sums);
        if (threadIdx.x == 0) *a.counter = 0u;
    }
}

// ---------------------------------------------------------------------------
// LDS-staged normal equations for the deep histories (8 < m <= 16).  The
// block loads each chunk of BLOCK points once (one point per thread,
// coalesced, non-temporal), forms the difference columns DF (and DX for
// PGR) and f there, and parks them in LDS; each of the four wavefronts then
// accumulates its quarter of the products over the chunk from LDS.  The
// next chunk's loads are issued before the current chunk's products, so
// HBM streams while they run, and HBM reads each needed ring slot once
// (the wavefront split of gram_split_kernel reads every slot once per
// wavefront, through L2).
// ---------------------------------------------------------------------------
template <typename T, int MM, int KIND>
struct GramLds {
    static constexpr int NC = (KIND == 1) ? 2 * MM + 1 : MM + 1;   // parked columns: DF, (DX), f
    static constexpr int LP = BLOCK;                             // points per chunk
};

template <typename T, int MM, int KIND, int W>
__device__ __forceinline__ void gram_lds_part(const GramArgs<T> &a, double (*sv)[BLOCK])
{
    using Ix = GramIdx<MM, KIND>;
    constexpr int NA = Ix::NA;
    constexpr int NS = MM + 1;
    constexpr int NC = GramLds<T, MM, KIND>::NC;
    constexpr int LP = GramLds<T, MM, KIND>::LP;
    constexpr int PER = (NA + BLOCK / 64 - 1) / (BLOCK / 64);
    constexpr int T0 = W * PER < NA ? W * PER : NA;
    constexpr int T1 = (W + 1) * PER < NA ? (W + 1) * PER : NA;
    constexpr int NT = T1 > T0 ? T1 - T0 : 1;
    const int nv = a.nvalid, dir = a.direct;
    const T *D = (KIND == 0) ? a.F : a.Y;
    const T *pd[NS], *px[NS];
    bool use[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        use[k] = dir ? (k < nv) : (k <= nv);
        const size_t off = (size_t)(use[k] ? a.slot[k] : 0) * a.ld;
        pd[k] = D + off;
        px[k] = a.F + off;
    }
    const T *pf = (KIND == 0 ? a.F : a.Y) + (size_t)a.fslot * a.ld;
    const bool f_is_d0 = !dir && a.fslot == a.slot[0];
    const long n = a.n;
    const long nch = (n + LP - 1) / LP;
    const int lane = threadIdx.x & 63;

    T rd[NS], rx[NS], rf = (T)0, rb = (T)0;
    auto load = [&](long c) {
        const long i = c * LP + threadIdx.x;
        const bool in = i < n;
#pragma unroll
        for (int k = 0; k < NS; k++) {
            rd[k] = (in && use[k]) ? __builtin_nontemporal_load(pd[k] + i) : (T)0;
            if constexpr (KIND == 1) rx[k] = (in && use[k]) ? __builtin_nontemporal_load(px[k] + i) : (T)0;
        }
        rf = in ? (f_is_d0 ? rd[0] : pf[i]) : (T)0;
        if constexpr (KIND != 0) rb = in ? a.b[i] : (T)0;
    };
    // the chunk's columns: DF = f - f_old (DX = x - x_old) by age, and f
    // (PGR.c:102-103: b - Ax), formed in T as the other Gram kernels do
    auto park = [&]() {
        const int t = threadIdx.x;
#pragma unroll
        for (int k = 0; k < MM; k++) {
            sv[k][t] = k < nv ? (dir ? (double)rd[k] : (double)(rd[k] - rd[k + 1])) : 0.0;
            if constexpr (KIND == 1) sv[MM + k][t] = k < nv ? (dir ? (double)rx[k] : (double)(rx[k] - rx[k + 1])) : 0.0;
        }
        if constexpr (KIND != 0) sv[NC - 1][t] = (double)(rb - rf);
        else sv[NC - 1][t] = (double)rf;
    };

    double acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = 0.0;
    long c = blockIdx.x;
    if (c < nch) load(c);
    for (; c < nch; c += gridDim.x) {
        park();
        __syncthreads();
        if (c + gridDim.x < nch) load(c + gridDim.x);
        if constexpr (T1 > T0) {
            for (int pp = lane; pp < LP; pp += 64) {
#pragma unroll
                for (int t = T0; t < T1; t++) {
                    const int j = Ix::j_of(t), q = Ix::q_of(t);
                    const double u = (q < 0) ? sv[NC - 1][pp] : (KIND == 1 ? sv[MM + (q < 0 ? 0 : q)][pp]
                                                                           : sv[q < 0 ? 0 : q][pp]);
                    const double v = (q < 0 && KIND == 1) ? sv[MM + j][pp] : sv[j][pp];
                    acc[t - T0] += u * v;
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = T0; t < T1; t++) {
        const double v = wave_sum(acc[t - T0]);
        if (lane == 0) a.partials[(size_t)t * a.nblocks + blockIdx.x] = v;
    }
}

template <typename T, int MM, int KIND>
__global__ __launch_bounds__(BLOCK) void gram_lds_kernel(const GramArgs<T> a)
{
    static_assert(BLOCK == 256, "four wavefronts share the products");
    constexpr int NA = GramIdx<MM, KIND>::NA;
    static_assert(NA <= GRAM_NA_MAX, "partials buffers hold GRAM_NA_MAX per block");
    __shared__ double sv[GramLds<T, MM, KIND>::NC][BLOCK];
    __shared__ double sums[NA];
    if (a.ctrl->done) return;
    switch (threadIdx.x >> 6) {
    case 0: gram_lds_part<T, MM, KIND, 0>(a, sv); break;
    case 1: gram_lds_part<T, MM, KIND, 1>(a, sv); break;
    case 2: gram_lds_part<T, MM, KIND, 2>(a, sv); break;
    default: gram_lds_part<T, MM, KIND, 3>(a, sv); break;
    }
    if (!a.counter) return;                     // two-pass: gram_finish_kernel follows
    if (last_block_arrive(a.counter, gridDim.x)) {
        final_sum_vm(a.partials, a.nblocks, NA, sums);
        gram_layout<T, MM, KIND>(a, sums);
        if (threadIdx.x == 0) *a.counter = 0u;
    }
}

template <typename T, int MM, int KIND, int NPASS, int PASS = 0>
void launch_split_passes(const GramArgs<T> &a, dim3 grid, dim3 block, hipStream_t st)
{
    hipLaunchKernelGGL((gram_split_kernel<T, MM, KIND, PASS, NPASS>), grid, block, 0, st, a);
    if constexpr (PASS + 1 < NPASS) launch_split_passes<T, MM, KIND, NPASS, PASS + 1>(a, grid, block, st);
}

template <typename T>
hipError_t launch_gram(const GramArgs<T> &a, hipStream_t st)
{
    if (a.m < 1 || a.m > MAXM || a.nvalid < 0 || a.nvalid > a.m) return hipErrorInvalidValue;
    if (a.kind < 0 || a.kind > 2) return hipErrorInvalidValue;
    dim3 grid(a.nblocks), block(BLOCK);
    // m <= 8: every accumulator in registers
    auto go = [&](auto c) {
        constexpr int M = decltype(c)::value;
        switch (a.kind) {
        case 0: hipLaunchKernelGGL((gram_kernel<T, M, 0>), grid, block, 0, st, a); break;
        case 1: hipLaunchKernelGGL((gram_kernel<T, M, 1>), grid, block, 0, st, a); break;
        default: hipLaunchKernelGGL((gram_kernel<T, M, 2>), grid, block, 0, st, a); break;
        }
    };
    auto go_lds = [&](auto c) {
        constexpr int M = decltype(c)::value;
        switch (a.kind) {
        case 0: hipLaunchKernelGGL((gram_lds_kernel<T, M, 0>), grid, block, 0, st, a); break;
        case 1: hipLaunchKernelGGL((gram_lds_kernel<T, M, 1>), grid, block, 0, st, a); break;
        default: hipLaunchKernelGGL((gram_lds_kernel<T, M, 2>), grid, block, 0, st, a); break;
        }
    };
    // 8 < m <= 16: the LDS-staged form, with an exact instantiation for the
    // READMEs' m = 13.  At 512^3, m = 13: AAR 2.63 ms against 2.91 ms with
    // every product in one thread's registers; PGR's square Gram 5.7 ms
    // against 10.9 ms split over wavefronts reading through L2
    if (a.kind == 0 && a.m == 7) {
        hipLaunchKernelGGL((gram_kernel<T, 7, 0>), grid, block, 0, st, a);
    } else if (a.m <= MAXM_FAST) {
        go(std::integral_constant<int, MAXM_FAST>());
    } else if (a.m == 13) {
        go_lds(std::integral_constant<int, 13>());
    } else if (a.m <= MAXM_MID) {
        go_lds(std::integral_constant<int, MAXM_MID>());
    } else {
        // 16 < m <= 32: 560 (AAR, PL2R) or 1056 (PGR) products, four and
        // eight passes of four slices, then the fixed-order finish
        switch (a.kind) {
        case 0: launch_split_passes<T, MAXM, 0, 4>(a, grid, block, st); break;
        case 1: launch_split_passes<T, MAXM, 1, 8>(a, grid, block, st); break;
        default: launch_split_passes<T, MAXM, 2, 4>(a, grid, block, st); break;
        }
    }
    return hipGetLastError();
}

template hipError_t launch_gram_solve<double>(const GramArgs<double> &, int, hipStream_t);
template hipError_t launch_gram_solve<float>(const GramArgs<float> &, int, hipStream_t);
template hipError_t launch_gram<double>(const GramArgs<double> &, hipStream_t);
template hipError_t launch_gram<float>(const GramArgs<float> &, hipStream_t);

}  // namespace aar
