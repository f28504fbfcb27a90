// helmholtz.hip -- complex Helmholtz kernels (no MPI_REAL counterpart; the
// AAR semantics follow MPI_REAL/AAR.c with the Hermitian Gram of
// PETSC_COMPLEX/AAR_Complex.c:207-246).
//
// Operator, complex128 interleaved (double2 = re, im), periodic:
//   A u = a*Lap(u) + (c(x) + i*eta) u,
// the Laplacian applied to re and im separately in the order of
// MPI_REAL/system.c:195-201, then y_re = lap_re + (c u_re - eta u_im),
// y_im = lap_im + (c u_im + eta u_re).  Jacobi: D = (a*3*coeff[0] + c) + i*eta,
// g = f / D computed as ((f_re D_re + f_im D_im) + i (f_im D_re - f_re D_im)) / |D|^2.
// The adjoint operator A^H is the same with eta -> -eta (the Laplacian is
// real symmetric and c real).
//
// The stencil keeps the design of stencil.hip (z-march with a register
// queue, LDS plane tile, XCD-aware tiles) on 16-byte points; its plane tile
// is twice as large, so halos are loaded per plane (no halo ring) and a
// thread owns two rows.  Small grids run one-shot boxes.
#include "aar_common.h"
#include "aar_device.h"
#include "aar_kernels.h"
#include "ls_body.h"

namespace aar {

namespace {

constexpr int HWY = 8;   // wavefronts per block (stacked in y)
constexpr int HPY = 2;   // rows per thread

__device__ inline int hmodp(int i, int n) { i %= n; return i < 0 ? i + n : i; }

__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(__dadd_rn(a.x, b.x), __dadd_rn(a.y, b.y)); }
__device__ inline double2 cscale(double2 a, double s) { return make_double2(__dmul_rn(a.x, s), __dmul_rn(a.y, s)); }

// (c + i eta) u added to the Laplacian part, in the oracle's order
__device__ inline double2 helm_diag_add(double2 lap, double2 u, double ck, double eta)
{
    const double tr = __dsub_rn(__dmul_rn(ck, u.x), __dmul_rn(eta, u.y));
    const double ti = __dadd_rn(__dmul_rn(ck, u.y), __dmul_rn(eta, u.x));
    return make_double2(__dadd_rn(lap.x, tr), __dadd_rn(lap.y, ti));
}

// f / D with D = dr + i di
__device__ inline double2 cdiv_d(double2 f, double dr, double di)
{
    const double den = __dadd_rn(__dmul_rn(dr, dr), __dmul_rn(di, di));
    const double re = __dadd_rn(__dmul_rn(f.x, dr), __dmul_rn(f.y, di)) / den;
    const double im = __dsub_rn(__dmul_rn(f.y, dr), __dmul_rn(f.x, di)) / den;
    return make_double2(re, im);
}

// What a sweep does with the Laplacian part lap of A u at one point (element
// g; ck = c(x), b the right-hand side): its output, and its norm term into acc.
template <HMode MODE>
__device__ __forceinline__ void helm_point(const HArgs &a, double2 lap, double2 u, double2 b, double ck, bool ok, int g,
                                           double &acc)
{
    const double eta = a.eta, om = a.omega;
    const double2 au = helm_diag_add(lap, u, ck, eta);
    const double dr = __dadd_rn(a.dlap, ck);
    if constexpr (MODE == HMode::MATVEC) {
        if (ok) a.out0[g] = au;
    } else if constexpr (MODE == HMode::TRUE_RES) {
        const double2 f = make_double2(__dsub_rn(b.x, au.x), __dsub_rn(b.y, au.y));
        acc += ok ? (f.x * f.x + f.y * f.y) : 0.0;
        if (ok) a.out0[g] = cdiv_d(f, dr, eta);
    } else {
        // g' = g - omega (A g)/D; |D g'|^2 = ||b - A x'||^2 at the point
        const double2 t = cdiv_d(au, dr, eta);
        const double2 gn = make_double2(__dsub_rn(u.x, __dmul_rn(om, t.x)), __dsub_rn(u.y, __dmul_rn(om, t.y)));
        if (ok) a.out0[g] = gn;
        if (a.trace) {
            const double den = dr * dr + eta * eta;
            acc += ok ? den * (gn.x * gn.x + gn.y * gn.y) : 0.0;
        }
    }
}

}  // namespace

template <HMode MODE>
__global__ __launch_bounds__(64 * HWY) void hstencil_kernel(const HArgs a)
{
    constexpr int WY = HWY, PY = HPY;
    constexpr int NT = 64 * WY;
    constexpr int TY = WY * PY;
    constexpr int LH = TY + 2 * R;
    constexpr int LW = TX + 2 * R;
    constexpr int NYH = (2 * R + WY - 1) / WY;
    constexpr int NXH = (2 * R * TY + NT - 1) / NT;
    constexpr int QN = 2 * R + 1;
    constexpr bool NEED_B = MODE == HMode::TRUE_RES;

    __shared__ double2 lds[2][LH][LW];
    __shared__ double red_scratch[8 * WY];

    if (a.ctrl && a.ctrl->done) return;

    const int item = xcd_item(blockIdx.x, a.nitems);
    const int itx = item % a.ntx;
    const int rest = item / a.ntx;
    const int ity = rest % a.nty;
    const int izc = rest / a.nty;
    const int x0 = itx * TX, y0 = ity * TY;
    const int z0 = izc * a.lz;
    const int z1 = min(z0 + a.lz, a.nz);
    const int tid = threadIdx.x, tx = tid & 63, ty = tid >> 6;
    const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = a.nxy;

    const int cx = hmodp(x0 + tx, nx);
    int c_off[PY];
    bool c_ok[PY];
#pragma unroll
    for (int p = 0; p < PY; p++) {
        const int y = y0 + ty * PY + p;
        c_off[p] = cx + hmodp(y, ny) * nx;
        c_ok[p] = (x0 + tx < nx) && (y < ny);
    }
    int yh_off[NYH], yh_row[NYH];
    bool yh_ok[NYH];
#pragma unroll
    for (int k = 0; k < NYH; k++) {
        const int hr0 = ty + WY * k;
        yh_ok[k] = hr0 < 2 * R;
        const int hr = yh_ok[k] ? hr0 : 0;
        const int gy = hr < R ? y0 - R + hr : y0 + TY + (hr - R);
        yh_off[k] = cx + hmodp(gy, ny) * nx;
        yh_row[k] = hr < R ? hr : TY + hr;
    }
    int xh_off[NXH], xh_row[NXH], xh_col[NXH];
    bool xh_ok[NXH];
#pragma unroll
    for (int k = 0; k < NXH; k++) {
        const int c = tid + NT * k;
        xh_ok[k] = c < 2 * R * TY;
        const int r = xh_ok[k] ? c / (2 * R) : 0, cc = xh_ok[k] ? c % (2 * R) : 0;
        const int gx = cc < R ? x0 - R + cc : x0 + TX + (cc - R);
        xh_off[k] = xh_ok[k] ? hmodp(gx, nx) + hmodp(y0 + r, ny) * nx : c_off[0];
        xh_row[k] = R + r;
        xh_col[k] = cc < R ? cc : TX + cc;
    }
    double wt[R + 1];
#pragma unroll
    for (int o = 0; o <= R; o++) wt[o] = a.w[o];

    double2 q[PY][QN];
    struct Pre {
        double2 qn[PY];
        double2 hy[NYH];
        double2 hx[NXH];
        double2 bb[PY];
        double cc[PY];
    };
    Pre s0, s1;

#pragma unroll
    for (int s = 0; s < 2 * R; s++) {
        const int zo = hmodp(z0 - R + s, nz) * nxy;
#pragma unroll
        for (int p = 0; p < PY; p++) q[p][s] = a.in0[c_off[p] + zo];
    }
    auto prefetch = [&](int zp, Pre &st) {
        const int zq = hmodp(zp + R, nz) * nxy, zc = hmodp(zp, nz) * nxy;
#pragma unroll
        for (int p = 0; p < PY; p++) st.qn[p] = a.in0[c_off[p] + zq];
#pragma unroll
        for (int k = 0; k < NYH; k++) st.hy[k] = a.in0[yh_off[k] + zc];
#pragma unroll
        for (int k = 0; k < NXH; k++) st.hx[k] = a.in0[xh_off[k] + zc];
#pragma unroll
        for (int p = 0; p < PY; p++) {
            if constexpr (NEED_B) st.bb[p] = a.bvec[c_off[p] + zc];
            st.cc[p] = a.c ? a.c[c_off[p] + zc] : a.c0;
        }
    };

    double acc = 0.0;
    auto plane = [&](const int z, Pre &cur, Pre &nxt) {
        const int buf = (z - z0) & 1;
#pragma unroll
        for (int p = 0; p < PY; p++) {
            q[p][2 * R] = cur.qn[p];
            lds[buf][R + ty * PY + p][R + tx] = q[p][R];
        }
#pragma unroll
        for (int k = 0; k < NYH; k++)
            if (yh_ok[k]) lds[buf][yh_row[k]][R + tx] = cur.hy[k];
#pragma unroll
        for (int k = 0; k < NXH; k++)
            if (xh_ok[k]) lds[buf][xh_row[k]][xh_col[k]] = cur.hx[k];
        prefetch(z + 1, nxt);
        __syncthreads();

        const int zoff = z * nxy;
#pragma unroll
        for (int p = 0; p < PY; p++) {
            const int lr = R + ty * PY + p, lc = R + tx;
            const double2 u = q[p][R];
            auto ynb = [&](int d) -> double2 {
                const int pp = p + d;
                if (pp >= 0 && pp < PY) return q[pp < 0 ? 0 : (pp < PY ? pp : PY - 1)][R];
                return lds[buf][lr + d][lc];
            };
            // system.c:195-201 order on each component
            double2 y = cscale(cscale(u, 3.0), wt[0]);
#pragma unroll
            for (int o = 1; o <= R; o++) {
                double2 nb = cadd(lds[buf][lr][lc - o], lds[buf][lr][lc + o]);
                nb = cadd(nb, ynb(-o));
                nb = cadd(nb, ynb(o));
                nb = cadd(nb, q[p][R - o]);
                nb = cadd(nb, q[p][R + o]);
                y = cadd(y, cscale(nb, wt[o]));
            }
            const double2 b = NEED_B ? cur.bb[p] : make_double2(0.0, 0.0);
            helm_point<MODE>(a, y, u, b, cur.cc[p], c_ok[p], c_off[p] + zoff, acc);
        }
#pragma unroll
        for (int p = 0; p < PY; p++)
#pragma unroll
            for (int s = 0; s < 2 * R; s++) q[p][s] = q[p][s + 1];
    };

    prefetch(z0, s0);
    int z = z0;
    for (; z + 1 < z1; z += 2) {
        plane(z, s0, s1);
        plane(z + 1, s1, s0);
    }
    if (z < z1) plane(z, s0, s1);

    if (a.partials) {
        double accv[1] = {acc};
        block_reduce_to<1, NT>(accv, a.partials + (size_t)item, red_scratch);
    }
}

// ---------------------------------------------------------------------------
// One-shot boxes for the smaller grids (see stencil_tile.h): 32 x 16 x LZ
// points a block, one column of LZ points a thread, all planes staged at once
// behind one barrier.  Bound by the chain of loads, one barrier and the 37
// ordered additions a block; at 96^3 (884736 points, 864 blocks of 8 waves)
// the recurrence sweep takes 15.5 us, the march 40 (its reads from HBM alone take
// 6).  A narrower 32 x 8 box
// loads 1.9 halo values a point against 1.1 (96^3 36.7 us with its update
// against 32.7).
// ---------------------------------------------------------------------------
constexpr int HBX = 32, HBY = 16, HBN = HBX * HBY;   // two rows a wavefront

template <HMode MODE, int LZ>
__global__ __launch_bounds__(HBN) void hstencil_box_kernel(const HArgs a)
{
    constexpr int NT = HBN, TY = HBY;
    constexpr int LH = TY + 2 * R, LW = HBX + 2 * R;
    constexpr int NYC = 2 * R * HBX, NXC = 2 * R * TY;
    constexpr int NHC = LZ * (NYC + NXC), NH = (NHC + NT - 1) / NT;
    constexpr int NQ = LZ + 2 * R;
    constexpr bool NEED_B = MODE == HMode::TRUE_RES;

    __shared__ double2 lds[LZ * LH][LW];
    __shared__ double red_scratch[NT / 64];

    if (a.ctrl && a.ctrl->done) return;

    const int item = xcd_item(blockIdx.x, a.nitems);
    const int itx = item % a.ntx;
    const int rest = item / a.ntx;
    const int x0 = itx * HBX, y0 = rest % a.nty * TY, z0 = rest / a.nty * LZ;
    const int tid = threadIdx.x, tx = tid % HBX, ty = tid / HBX;
    const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = a.nxy;

    const unsigned c_off = (unsigned)(hmodp(x0 + tx, nx) + hmodp(y0 + ty, ny) * nx);
    const bool c_ok = (x0 + tx < nx) && (y0 + ty < ny);
    size_t zo[NQ];                                   // planes z0-R .. z0+LZ-1+R (wrapped; uniform)
    {
        int z = hmodp(z0 - R, nz);
#pragma unroll
        for (int s = 0; s < NQ; s++) {
            zo[s] = (size_t)z * nxy;
            z = z + 1 == nz ? 0 : z + 1;
        }
    }
    double2 q[NQ];
#pragma unroll
    for (int s = 0; s < NQ; s++) q[s] = (a.in0 + zo[s])[c_off];
    // halo cell c of the box: plane, then 2R rows of HBX, then TY rows of R
    // left and R right
    double2 h[NH];
    int h_row[NH], h_col[NH];
#pragma unroll
    for (int j = 0; j < NH; j++) {
        const int c0 = tid + NT * j;
        const int cc = c0 < NHC ? c0 : 0;
        const int s = cc / (NYC + NXC), c = cc % (NYC + NXC);
        int gx, gy;
        if (c < NYC) {
            const int r = c / HBX, w = c % HBX;
            gx = x0 + w;
            gy = r < R ? y0 - R + r : y0 + TY + (r - R);
            h_row[j] = s * LH + (r < R ? r : TY + r);
            h_col[j] = R + w;
        } else {
            const int r = (c - NYC) / (2 * R), w = (c - NYC) % (2 * R);
            gx = w < R ? x0 - R + w : x0 + HBX + (w - R);
            gy = y0 + r;
            h_row[j] = s * LH + R + r;
            h_col[j] = w < R ? w : HBX + w;
        }
        h[j] = a.in0[(unsigned)(hmodp(gx, nx) + hmodp(gy, ny) * nx) + (unsigned)hmodp(z0 + s, nz) * (unsigned)nxy];
    }
    double2 bb[LZ];
    double ck[LZ];
#pragma unroll
    for (int s = 0; s < LZ; s++) {
        if constexpr (NEED_B) bb[s] = (a.bvec + zo[R + s])[c_off];
        ck[s] = a.c ? (a.c + zo[R + s])[c_off] : a.c0;
    }
#pragma unroll
    for (int s = 0; s < LZ; s++) lds[s * LH + R + ty][R + tx] = q[R + s];
#pragma unroll
    for (int j = 0; j < NH; j++)
        if (tid + NT * j < NHC) lds[h_row[j]][h_col[j]] = h[j];
    __syncthreads();

    double acc = 0.0;
#pragma unroll
    for (int s = 0; s < LZ; s++) {
        if (z0 + s < nz) {                           // uniform: planes past the grid
            const int lr = s * LH + R + ty, lc = R + tx;
            const double2 u = q[R + s];
            // system.c:195-201 order on each component
            double2 y = cscale(cscale(u, 3.0), a.w[0]);
#pragma unroll
            for (int o = 1; o <= R; o++) {
                double2 nb = cadd(lds[lr][lc - o], lds[lr][lc + o]);
                nb = cadd(nb, lds[lr - o][lc]);
                nb = cadd(nb, lds[lr + o][lc]);
                nb = cadd(nb, q[R + s - o]);
                nb = cadd(nb, q[R + s + o]);
                y = cadd(y, cscale(nb, a.w[o]));
            }
            const double2 b = NEED_B ? bb[s] : make_double2(0.0, 0.0);
            helm_point<MODE>(a, y, u, b, ck[s], c_ok, (int)(c_off + zo[R + s]), acc);
        }
    }
    if (a.partials) {
        double accv[1] = {acc};
        block_reduce_to<1, NT>(accv, a.partials + (size_t)item, red_scratch);
    }
}

// Where the boxes are faster than the march (recurrence sweep, its norm's
// finish and a one-vector update, microseconds, march / boxes): 24^3 44.1 /
// 12.8, 48^3 46.3 / 14.5, 64^3 48.2 / 15.9, 96^3 57.6 / 32.7, 128^3 72.6 /
// 62.2, 144^3 84.6 / 89.6, 160^3 106 / 114, 256^3 379 / 435: the march's deep
// columns leave most CUs idle on the small grids, the boxes' (LZ + 12)/LZ
// reads a point cost more on the large ones.  Boxes of 2 planes while those of
// 4 are one a CU or fewer (64^3 18.2 -> 15.9, 96^3 32.7 -> 34.3).
static void hgeometry(HArgs &a)
{
    a.nxy = a.nx * a.ny;
    a.box = 0;
    if (a.lz <= 0 && (long)a.nxy * a.nz <= 2500000L) {
        const int tx = (a.nx + HBX - 1) / HBX, ty = (a.ny + HBY - 1) / HBY;
        a.box = (long)tx * ty * ((a.nz + 3) / 4) <= 256 ? 2 : 4;
        a.lz = a.box;
        a.ntx = tx;
        a.nty = ty;
        a.nzc = (a.nz + a.lz - 1) / a.lz;
        a.nitems = a.ntx * a.nty * a.nzc;
        return;
    }
    a.ntx = (a.nx + TX - 1) / TX;
    a.nty = (a.ny + HWY * HPY - 1) / (HWY * HPY);
    if (a.lz <= 0) {
        const int cols = a.ntx * a.nty;
        int nzc = std::max(1, 256 / std::max(1, cols));
        int lz = (a.nz + nzc - 1) / nzc;
        a.lz = std::max(lz, std::min(a.nz, 16));
    }
    if (a.lz > a.nz) a.lz = a.nz;
    a.nzc = (a.nz + a.lz - 1) / a.lz;
    a.nitems = a.ntx * a.nty * a.nzc;
}

int hstencil_items(const HArgs &a0)
{
    HArgs a = a0;
    hgeometry(a);
    return a.nitems;
}

template <HMode M> static void launch_hsweep(const HArgs &a, hipStream_t st)
{
    const dim3 grid(a.nitems);
    if (a.box == 2) hipLaunchKernelGGL((hstencil_box_kernel<M, 2>), grid, dim3(HBN), 0, st, a);
    else if (a.box == 4) hipLaunchKernelGGL((hstencil_box_kernel<M, 4>), grid, dim3(HBN), 0, st, a);
    else hipLaunchKernelGGL((hstencil_kernel<M>), grid, dim3(64 * HWY), 0, st, a);
}

hipError_t launch_hstencil(HMode m, const HArgs &a0, hipStream_t st)
{
    HArgs a = a0;
    hgeometry(a);
    switch (m) {
    case HMode::MATVEC: launch_hsweep<HMode::MATVEC>(a, st); break;
    case HMode::TRUE_RES: launch_hsweep<HMode::TRUE_RES>(a, st); break;
    case HMode::REC: launch_hsweep<HMode::REC>(a, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Hermitian Gram of the complex g ring (PETSC_COMPLEX/AAR_Complex.c:213-236)
// ---------------------------------------------------------------------------
template <int MM>
__global__ __launch_bounds__(BLOCK) void hgram_kernel(const HGramArgs a)
{
    constexpr int NG = MM * (MM + 1) / 2;
    constexpr int NA = 2 * (NG + MM);
    static_assert(NA <= HGRAM_NA_MAX, "partials buffers hold HGRAM_NA_MAX per block");
    constexpr int NS = MM + 1;
    __shared__ double scratch[NA * (BLOCK / 64)];
    if (a.ctrl->done) return;
    const int nv = a.nvalid;
    const double2 *pd[NS];
    bool use[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        use[k] = k <= nv;
        pd[k] = a.F + (size_t)(use[k] ? a.slot[k] : 0) * a.ld;
    }
    double acc[NA];
#pragma unroll
    for (int k = 0; k < NA; k++) acc[k] = 0.0;
    const long stride = (long)gridDim.x * BLOCK;
    for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < a.n; i += stride) {
        double2 v[NS];
#pragma unroll
        for (int k = 0; k < NS; k++)
            v[k] = use[k] ? ld_nt2<double2>(reinterpret_cast<const double *>(pd[k] + i)) : make_double2(0.0, 0.0);
        double dr[MM], di[MM];
#pragma unroll
        for (int k = 0; k < MM; k++) {
            dr[k] = k < nv ? v[k].x - v[k + 1].x : 0.0;     // DF = f - f_old
            di[k] = k < nv ? v[k].y - v[k + 1].y : 0.0;
        }
        const double fr = v[0].x, fi = v[0].y;
        int t = 0;
#pragma unroll
        for (int j = 0; j < MM; j++) {
#pragma unroll
            for (int q = 0; q <= j; q++) {
                // <DF_q, DF_j> = conj(DF_q) DF_j
                acc[2 * t] += dr[q] * dr[j] + di[q] * di[j];
                acc[2 * t + 1] += dr[q] * di[j] - di[q] * dr[j];
                t++;
            }
            acc[2 * NG + 2 * j] += dr[j] * fr + di[j] * fi;       // <DF_j, f>
            acc[2 * NG + 2 * j + 1] += dr[j] * fi - di[j] * fr;
        }
    }
    // value-major partials: each value's per-block sums are contiguous
    block_reduce_to_vm<NA>(acc, a.partials + blockIdx.x, a.nblocks, scratch);
}

// One block: fixed-order sums of the partials (one wavefront per value), the
// real 2m x 2m system E = [Gr -Gi; Gi Gr] (E[i][j] at G[j*n + i], rhs at
// G[n*n + i], n = 2m) with every thread laying out its entries, and its solve
// by the first wavefront.
template <int M2> constexpr int HFIN_NT = M2 <= 16 ? 512 : 256;

template <int MM, int M2>
__global__ __launch_bounds__(HFIN_NT<M2>) void hgram_finish_kernel(const HGramArgs a)
{
    constexpr int NG = MM * (MM + 1) / 2;
    constexpr int NA = 2 * (NG + MM);
    static_assert(M2 >= 2 * MM, "the embedded system fits");
    __shared__ double sums[NA];
    __shared__ LsLds<M2> L;
    if (a.ctrl->done) return;
    final_sum_vm<HFIN_NT<M2>>(a.partials, a.nblocks, NA, sums);
    const int m = a.m, n2 = 2 * m, nv = a.nvalid;
    // age of the reference's column c (ages as in GramArgs)
    auto age = [&](int c) { return ((a.it - 2 - c) % m + m) % m; };
    auto entry = [&](int e) -> double {
        if (e >= n2 * n2) {
            const int r = e - n2 * n2, k = age(r % m);
            return k < nv ? sums[2 * NG + 2 * k + r / m] : 0.0;
        }
        const int i = e % n2, j = e / n2;                  // E[i][j]
        const int ki = age(i % m), kj = age(j % m);
        if (ki >= nv || kj >= nv) return 0.0;
        // <DF_q, DF_p> of ages q <= p at p(p+1)/2 + q: Gr[i][j] = re, Gi[i][j]
        // = im for i of age q, the conjugate for the other order
        const int p = ki > kj ? ki : kj, q = ki > kj ? kj : ki;
        const double re = sums[2 * (p * (p + 1) / 2 + q)];
        double im = sums[2 * (p * (p + 1) / 2 + q) + 1];
        if (ki >= kj) im = -im;
        const int bi = i / m, bj = j / m;
        return bi == bj ? re : (bi == 0 ? -im : im);
    };
    for (int e = threadIdx.x; e < n2 * n2 + n2; e += HFIN_NT<M2>) {
        const double v = entry(e);
        a.ctrl->G[e] = v;
        if (e < n2 * n2) L.A[e % n2][e / n2] = v;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x;
    ls_solve<M2>(L, lane < n2 ? entry(n2 * n2 + lane) : 0.0, a.ctrl, n2, a.flags);
}

hipError_t launch_hgram(const HGramArgs &a, hipStream_t st)
{
    if (a.m < 1 || a.m > MAXM_CPLX || 2 * a.m > MAXM_LS || a.nvalid < 0 || a.nvalid > a.m) return hipErrorInvalidValue;
    const dim3 grid(a.nblocks), block(BLOCK);
    // deeper histories (the reference's complex README run uses m = 13): 304
    // accumulators, partly spilled; correct, at lower throughput
    if (a.m <= 7) hipLaunchKernelGGL((hgram_kernel<7>), grid, block, 0, st, a);
    else if (a.m <= 8) hipLaunchKernelGGL((hgram_kernel<8>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((hgram_kernel<MAXM_CPLX>), grid, block, 0, st, a);
    return hipGetLastError();
}

hipError_t launch_hgram_solve(const HGramArgs &a, hipStream_t st)
{
    const dim3 grid(1);
    if (a.m <= 7) hipLaunchKernelGGL((hgram_finish_kernel<7, 16>), grid, dim3(HFIN_NT<16>), 0, st, a);
    else if (a.m <= 8) hipLaunchKernelGGL((hgram_finish_kernel<8, 16>), grid, dim3(HFIN_NT<16>), 0, st, a);
    else hipLaunchKernelGGL((hgram_finish_kernel<MAXM_CPLX, 2 * MAXM_CPLX>), grid, dim3(HFIN_NT<32>), 0, st, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// complex anchor update (see HAncArgs / AncArgs).  ONE (histories up to 8):
// one element per thread and one block per BLOCK elements, x read and
// written non-temporally, as the FP64 real update.  The deeper form keeps a
// grid stride over at most 4096 blocks (its registers leave too few waves
// for one element per thread, as measured for the real update).
// ---------------------------------------------------------------------------
template <int NGM, int NCM, bool ONE>
__global__ __launch_bounds__(BLOCK) void hanchor_update_kernel(const HAncArgs a)
{
    __shared__ double s_cg[2 * NGMAX], s_cc[2 * NCMAX];
    if (a.ctrl && a.ctrl->done) return;
    if (threadIdx.x == 0) {
        for (int i = 0; i < NGMAX; i++) {
            s_cg[2 * i] = (a.with_beta && i == a.ng - 1) ? a.beta : 0.0;
            s_cg[2 * i + 1] = 0.0;
        }
        for (int c = 0; c < 2 * NCMAX; c++) s_cc[c] = 0.0;
        for (int t = 0; t < a.ncol; t++) {
            const double gr = a.ctrl->s[a.col_ref[t]], gi = a.ctrl->s[a.m + a.col_ref[t]];
            const int j = a.col_j[t], cj = a.col_c[t];
            s_cg[2 * j] -= a.beta * gr;
            s_cg[2 * j + 1] -= a.beta * gi;
            const double f = (cj < 0) ? (a.beta - a.omega) : a.beta;
            s_cg[2 * (j - 1)] += f * gr;
            s_cg[2 * (j - 1) + 1] += f * gi;
            if (cj >= 0) {
                s_cc[2 * cj] -= gr;
                s_cc[2 * cj + 1] -= gi;
            }
        }
    }
    __syncthreads();
    const int ng = a.ng, nc = a.nc;
    double2 *co = (a.cout >= 0) ? a.C + (size_t)a.cout * a.ld : nullptr;
    const long stride = ONE ? a.n : (long)gridDim.x * BLOCK;
    for (long e = (long)blockIdx.x * BLOCK + threadIdx.x; e < a.n; e += stride) {
        double sxr = 0.0, sxi = 0.0, scr = 0.0, sci = 0.0;
        // every stream's load issued before the sums (static slot indices)
        double2 gv[NGM], cv[NCM];
#pragma unroll
        for (int i = 0; i < NGM; i++)
            if (i < ng) gv[i] = ld_nt2<double2>(reinterpret_cast<const double *>(a.G + (size_t)a.gslot[i] * a.ld + e));
#pragma unroll
        for (int c = 0; c < NCM; c++)
            if (c < nc) cv[c] = ld_nt2<double2>(reinterpret_cast<const double *>(a.C + (size_t)a.cslot[c] * a.ld + e));
#pragma unroll
        for (int i = 0; i < NGM; i++)
            if (i < ng) {
                const double2 g = gv[i];
                if (i >= a.xlo && i < a.xhi) {
                    sxr += g.x;
                    sxi += g.y;
                }
                const double cr = s_cg[2 * i], ci = s_cg[2 * i + 1];
                scr += cr * g.x - ci * g.y;
                sci += cr * g.y + ci * g.x;
            }
#pragma unroll
        for (int c = 0; c < NCM; c++)
            if (c < nc) {
                const double2 v = cv[c];
                const double cr = s_cc[2 * c], ci = s_cc[2 * c + 1];
                scr += cr * v.x - ci * v.y;
                sci += cr * v.y + ci * v.x;
            }
        if (ONE) {
            const double2 xv = ld_nt2<double2>(reinterpret_cast<const double *>(a.x + e));
            st_nt2(reinterpret_cast<double *>(a.x + e),
                   make_double2(xv.x + (a.omega * sxr + scr), xv.y + (a.omega * sxi + sci)));
        } else {
            const double2 xv = a.x[e];
            a.x[e] = make_double2(xv.x + (a.omega * sxr + scr), xv.y + (a.omega * sxi + sci));
        }
        if (co) st_nt2(reinterpret_cast<double *>(co + e), make_double2(scr, sci));
    }
}

hipError_t launch_hanchor_update(const HAncArgs &a, hipStream_t st)
{
    constexpr int HNG = MAXM_CPLX + 2, HNC = MAXM_CPLX + 1;   // the complex solver's m <= 16
    if (a.ng < 1 || a.ng > HNG || a.nc < 0 || a.nc > HNC || a.ncol < 0 || a.ncol > MAXM_CPLX)
        return hipErrorInvalidValue;
    if (a.xlo < 0 || a.xhi > a.ng || !a.G || !a.x) return hipErrorInvalidValue;
    if ((a.nc > 0 || a.cout >= 0) && !a.C) return hipErrorInvalidValue;
    if (a.ncol > 0 && !a.ctrl) return hipErrorInvalidValue;
    for (int t = 0; t < a.ncol; t++)
        if (a.col_j[t] < 1 || a.col_j[t] >= a.ng || a.col_c[t] >= a.nc || a.col_ref[t] < 0 ||
            a.col_ref[t] >= a.m)
            return hipErrorInvalidValue;
    long nb = (a.n + BLOCK - 1) / BLOCK;
    if (nb < 1) nb = 1;
    if (nb > 0x7fffffffL) return hipErrorInvalidValue;
    const long nstride = std::min(nb, 4096L);
    // histories up to 8 (an (8, 1) form with half the registers measured 4%
    // slower at 256^3), and the deeper ones
    if (a.ng <= MAXM_FAST + 2 && a.nc <= MAXM_FAST + 1)
        hipLaunchKernelGGL((hanchor_update_kernel<MAXM_FAST + 2, MAXM_FAST + 1, true>), dim3((unsigned)nb), dim3(BLOCK),
                           0, st, a);
    else
        hipLaunchKernelGGL((hanchor_update_kernel<HNG, HNC, false>), dim3((unsigned)nstride), dim3(BLOCK), 0, st, a);
    return hipGetLastError();
}

// dL/dc_k = -Re(conj(lambda_k) u_k)
__global__ __launch_bounds__(BLOCK) void helm_grad_c_kernel(long n, const double2 *lam, const double2 *u, double *dc)
{
    const long stride = (long)gridDim.x * BLOCK;
    for (long e = (long)blockIdx.x * BLOCK + threadIdx.x; e < n; e += stride) {
        const double2 l = lam[e], v = u[e];
        dc[e] = -(l.x * v.x + l.y * v.y);
    }
}

hipError_t launch_helm_grad_c(long n, const double2 *lambda, const double2 *u, double *dc, hipStream_t st)
{
    if (n < 1 || !lambda || !u || !dc) return hipErrorInvalidValue;
    long nb = (n + BLOCK - 1) / BLOCK;
    nb = nb < 1 ? 1 : (nb > 8192 ? 8192 : nb);
    hipLaunchKernelGGL(helm_grad_c_kernel, dim3((unsigned)nb), dim3(BLOCK), 0, st, n, lambda, u, dc);
    return hipGetLastError();
}

}  // namespace aar
