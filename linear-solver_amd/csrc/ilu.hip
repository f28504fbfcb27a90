// ilu.hip -- ILU(0) of the periodic FD12 star matrix (the PETSc variant's
// pc = 1: PCBJACOBI -> PCILU on one block, PETSC_REAL/main.c:88-91; PCICC of
// AAR_Real.c:58-60 is the same preconditioner in exact arithmetic on this
// symmetric matrix), and its complex form.
//
// Every dependency of a row (x, y, z) in the elimination and in the forward
// solve has a smaller x + y + z (periodic wrap included).  Rows are eliminated
// in PETSc's IKJ order and solved in ascending column order, with no sums
// across rows: the factors and solves are bit-identical to the oracle's
// sequential ones.
//
// The grid is cut into 8^3 tiles, whose own dependencies go to tiles of a
// smaller ti + tj + tk: one launch per tile diagonal (3 n/8 - 2 of them), one
// wavefront per tile.  Lane = (x, y) of the tile, which walks its z-column
// skewed, one level x + y + z after the other (22 levels), so the levels of a
// tile follow each other without a launch or a block barrier, and the solved
// values of the tile pass from level to level in LDS.  A launch per level of
// the whole grid (3 n - 2 of them, each a chain of scattered loads) took
// 6.6-7.8 us a level, 2.4 ms an apply at 64^3; this form takes 17 us a tile
// diagonal, 0.75 ms an apply, and the factorization 7.7 -> 3.6 ms.  (Prefetching
// the rows level by level from memory instead of staging them: 38 us a
// diagonal.)
//
// What bounds it: the chain of 18 ordered subtractions a level and the LDS
// reads that feed it.
//
// Factor layout: value s of all rows is contiguous (s = 0: 1/u_ii; 1 + 12*axis
// + k the entry at periodic offset d along axis, k = d + 6 for d < 0, d + 5
// for d > 0: l_ij below the row, u_ij above), tile by tile, a tile's 512 rows
// in [z][y][x] order.
#include "ilu.h"

#include <algorithm>
#include <type_traits>

namespace aar {

namespace {

constexpr int TS = ILU_TS, NL = 3 * TS - 2;

__host__ __device__ constexpr int islot(int ax, int d) { return 1 + 12 * ax + (d < 0 ? d + 6 : d + 5); }

// periodic offsets of a row's columns along one axis in ascending column
// order: q = 0..5 -> d = 1..6 (below the row only when wrapped), q = 6..11
// -> d = -6..-1 (below unless wrapped)
__device__ __forceinline__ constexpr int qoff(int q) { return q < 6 ? q + 1 : q - 12; }

// scalar operations of the real and complex factorizations (complex:
// explicit formulas, as the oracle's)
__device__ __forceinline__ double s_mul(double a, double b) { return a * b; }
__device__ __forceinline__ double2 s_mul(double2 a, double2 b)
{
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double s_sub(double a, double b) { return a - b; }
__device__ __forceinline__ double2 s_sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double s_sel(bool c, double a, double b) { return c ? a : b; }
__device__ __forceinline__ double2 s_sel(bool c, double2 a, double2 b)
{
    return make_double2(c ? a.x : b.x, c ? a.y : b.y);
}
__device__ __forceinline__ double s_inv(double a) { return 1.0 / a; }
__device__ __forceinline__ double2 s_inv(double2 b)
{
    const double den = b.x * b.x + b.y * b.y;
    return make_double2((1.0 * b.x + 0.0 * b.y) / den, (0.0 * b.x - 1.0 * b.y) / den);
}
template <typename T> __device__ __forceinline__ T s_make(double re, double im);
template <> __device__ __forceinline__ double s_make<double>(double re, double) { return re; }
template <> __device__ __forceinline__ double2 s_make<double2>(double re, double im) { return make_double2(re, im); }

// the tile grid and the position of a row's values
struct TileMap {
    int tx, ty, tz;
    size_t np;                       // rows, padded to whole tiles
    __host__ __device__ TileMap(int nx, int ny, int nz)
        : tx((nx + TS - 1) / TS), ty((ny + TS - 1) / TS), tz((nz + TS - 1) / TS), np((size_t)tx * ty * tz * ILU_TP)
    {
    }
    __device__ __forceinline__ size_t row(int x, int y, int z) const
    {
        const size_t t = ((size_t)(z / TS) * ty + y / TS) * tx + x / TS;
        return t * ILU_TP + ((z % TS) * TS + y % TS) * TS + x % TS;
    }
};

// this block's tile on the launch's diagonal, or false
template <typename T>
__device__ __forceinline__ bool ilu_tile(const IluArgsT<T> &a, const TileMap &m, int &ti, int &tj, int &tk)
{
    ti = a.t0x + blockIdx.x % a.wx;
    tj = a.t0y + blockIdx.x / a.wx;
    tk = a.diag_tiles - ti - tj;
    return tk >= 0 && tk < m.tz;
}

}  // namespace

// ---------------------------------------------------------------------------
// factorization: the rows of one tile
// ---------------------------------------------------------------------------

// Row i's elimination on one axis by the rows k of it below i (IKJ: k in
// ascending order): l_ik = v_ik / u_kk, then v_ij -= l_ik u_kj for the columns
// j > k of both rows, which lie on this axis.  v: row i's values.  c, n: i's
// coordinate and the side.  row(ck): the values of the row at coordinate ck.
// ANY: sides of at least 13; else of at least 3R + 1, where two columns of a
// pattern are never closer across the boundary than inside it, so that the
// offset of j from k is d_ij - d_ik, the entries taken from k are known at
// compile time, and all of them are loaded before the chain starts (a level
// takes one memory latency an axis, not one a k).
template <typename T, int AX, bool ANY, typename Row>
__device__ __forceinline__ void ilu_eliminate(T (&v)[ILU_ROW], const int c, const int n, const size_t np, const bool lo,
                                              const bool hi, Row row)
{
    if constexpr (ANY) {
        for (int q = 0; q < 12; q++) {
            const int dk = qoff(q);
            const bool lower = dk > 0 ? (c + dk >= n) : (c + dk >= 0);
            if (!lower) continue;
            const int ck = dk > 0 ? c + dk - n : c + dk;
            const T *Fk = row(ck);
            const T l = s_mul(v[islot(AX, dk)], Fk[0]);
            v[islot(AX, dk)] = l;
            // row k's columns above k that are in row i's pattern: on this axis
            for (int dij = -R; dij <= R; dij++) {
                if (dij == dk) continue;
                int cj = c + dij;
                cj = cj < 0 ? cj + n : (cj >= n ? cj - n : cj);
                if (cj <= ck) continue;
                int dkj = dij - dk;
                if (dkj > R) dkj -= n;
                else if (dkj < -R) dkj += n;
                if (dkj < -R || dkj > R) continue;
                const int si = dij == 0 ? 0 : islot(AX, dij);
                v[si] = s_sub(v[si], s_mul(l, Fk[(size_t)islot(AX, dkj) * np]));
            }
        }
    } else {
        // the rows at d_ik = D0 .. D0 + 5; W: across the boundary
        auto rows = [&](auto w, const bool edge) {
            constexpr bool W = decltype(w)::value;
            constexpr int D0 = W ? 1 : -R;
            T f0[R], up[R][R], dn[R][R];
            bool ok[R];
#pragma unroll
            for (int a = 0; a < R; a++) {
                const int ck = W ? c + D0 + a - n : c + D0 + a;
                ok[a] = ck >= 0;
                const T *Fk = row(ok[a] ? ck : c);
                f0[a] = Fk[0];
#pragma unroll
                for (int e = 1; e <= R; e++) {
                    if (D0 + a + e <= R) up[a][e - 1] = Fk[(size_t)islot(AX, e) * np];
                    if (D0 + a - e >= -R && edge) dn[a][e - 1] = Fk[(size_t)islot(AX, -e) * np];
                }
            }
#pragma unroll
            for (int a = 0; a < R; a++) {
                const int dk = D0 + a;
                const T l = s_mul(v[islot(AX, dk)], f0[a]);
                v[islot(AX, dk)] = s_sel(ok[a], l, v[islot(AX, dk)]);
#pragma unroll
                for (int dij = -R; dij <= R; dij++) {
                    const int dkj = dij - dk;
                    if (dkj == 0 || dkj < -R || dkj > R) continue;
                    if (dkj < 0 && !edge) continue;
                    // j above k: for d_ij > d_ik unless j wraps to the low end
                    // (k does too when W); else where j lies across the
                    // boundary from k
                    const bool in = ok[a] && (dkj > 0 ? (W || c + dij < n) : (W ? c + dij < n : c + dij < 0));
                    const int si = dij == 0 ? 0 : islot(AX, dij);
                    const T u = dkj > 0 ? up[a][dkj > 0 ? dkj - 1 : 0] : dn[a][dkj < 0 ? -dkj - 1 : 0];
                    v[si] = s_sel(in, s_sub(v[si], s_mul(l, u)), v[si]);
                }
            }
        };
        if (hi) rows(std::true_type{}, true);
        if (lo) rows(std::false_type{}, true);
        else rows(std::false_type{}, false);
    }
}

template <typename T, bool ANY>
__global__ __launch_bounds__(64) void ilu_factor_kernel(const IluArgsT<T> a)
{
    const TileMap m(a.nx, a.ny, a.nz);
    int ti, tj, tk;
    if (!ilu_tile(a, m, ti, tj, tk)) return;
    const int lx = threadIdx.x % TS, ly = threadIdx.x / TS;
    const int x = ti * TS + lx, y = tj * TS + ly;
    for (int L = 0; L < NL; L++) {
        const int lz = L - lx - ly, z = tk * TS + lz;
        if (lz >= 0 && lz < TS && x < a.nx && y < a.ny && z < a.nz) {
            const size_t i = x + (size_t)y * a.nx + (size_t)z * a.nx * a.ny;
            T v[ILU_ROW];
            v[0] = s_make<T>(a.c ? a.diag + a.c[i] : a.diag, a.eta);
#pragma unroll
            for (int ax = 0; ax < 3; ax++)
#pragma unroll
                for (int d = 1; d <= R; d++) {
                    v[islot(ax, -d)] = s_make<T>(a.w[d], 0.0);
                    v[islot(ax, d)] = s_make<T>(a.w[d], 0.0);
                }
            // z, y, x: ascending column index
            ilu_eliminate<T, 2, ANY>(v, z, a.nz, m.np, tk == 0, tk * TS + TS > a.nz - R,
                                     [&](int ck) { return a.F + m.row(x, y, ck); });
            ilu_eliminate<T, 1, ANY>(v, y, a.ny, m.np, tj == 0, tj * TS + TS > a.ny - R,
                                     [&](int ck) { return a.F + m.row(x, ck, z); });
            ilu_eliminate<T, 0, ANY>(v, x, a.nx, m.np, ti == 0, ti * TS + TS > a.nx - R,
                                     [&](int ck) { return a.F + m.row(ck, y, z); });
            T *Fi = a.F + m.row(x, y, z);
            Fi[0] = s_inv(v[0]);
#pragma unroll
            for (int s = 1; s < ILU_ROW; s++) Fi[(size_t)s * m.np] = v[s];
        }
        // the level's rows are read by the next ones of this wavefront
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
    }
}

// ---------------------------------------------------------------------------
// triangular solve of one tile, in place on io (in -> io when in != io at the
// first solve of an apply).  LOWER: the columns below the row (tiles and
// levels upwards), else above (downwards); TRANS: the transposed factor
// (entries of the other row); DIAG: multiply by 1/u_ii at the end.
//
// Four wavefronts load everything the tile needs into LDS at once (one memory
// latency a tile; with the entries loaded level by level, even one level
// ahead, each level waited for memory: 38 us a launch); then one wavefront
// walks the levels from LDS.  Of a level's 18 products all but the 3 with the
// level just before are made a level ahead, so a level is its chain of
// subtractions and little else.
// ---------------------------------------------------------------------------
constexpr int ILU_NT = 256;

template <typename T, bool LOWER, bool TRANS, bool DIAG>
__global__ __launch_bounds__(ILU_NT) void ilu_solve_kernel(const IluArgsT<T> a, const T *in, T *io)
{
    constexpr int H = R, LP = TS + H + 1;        // a line of the tile with its halo, odd pitch
    constexpr int C0 = LOWER ? H : 0;            // tile cell 0 of a line
    constexpr int HB = LOWER ? 0 : TS;           // the halo's R cells
    constexpr int J1 = LOWER ? R - 1 : 0;        // of the R columns of an axis, the one next to the row
    // The factor rows are staged in whole (real), by [z][y][x], or (complex:
    // 160 kB of LDS) in two halves of 11 levels and 256 rows, in level order.
    constexpr int NCH = (int)(sizeof(T) / 8), CR = ILU_TP / NCH, LCH = NL / NCH;
    constexpr bool WST = sizeof(T) == 8;         // stage the entries across the boundary too
    constexpr int NT3 = R * (R + 1) / 2;         // those of a line
    constexpr int NSL = 3 * R + (DIAG ? 1 : 0);
    __shared__ T fs[NSL][CR];
    __shared__ T wf[3][WST ? TS * TS * NT3 : 1];
    // the tile's values by lines along x ([z][y]), y ([z][x]) and z ([y][x]),
    // and the R values across the periodic boundary of each line
    __shared__ T ln[3][TS * TS][LP];
    __shared__ T wr[3][TS * TS][R];
    __shared__ unsigned char plc[NCH == 1 ? 1 : ILU_TP];         // place() of a row by [z][y][x]
    const int skip = *a.skip;                    // looked at once the loads are under way
    const TileMap m(a.nx, a.ny, a.nz);
    int tc[3];
    if (!ilu_tile(a, m, tc[0], tc[1], tc[2])) return;
    const int tid = threadIdx.x, lane = tid & 63, lx = lane % TS, ly = lane / TS;
    const int dims[3] = {a.nx, a.ny, a.nz};
    const size_t st[3] = {1, (size_t)a.nx, (size_t)a.nx * a.ny};
    const size_t tile = (((size_t)tc[2] * m.ty + tc[1]) * m.tx + tc[0]) * ILU_TP;
    const T zero = s_make<T>(0.0, 0.0);
    // rows across the boundary: c + d >= n (below) for c >= n - R, c + d < 0
    // (above) for c < R.  own: 13 points, where such a column can lie in this
    // tile; its value is then the one solved here
    bool wrap[3], own[3];
#pragma unroll
    for (int ax = 0; ax < 3; ax++) {
        wrap[ax] = LOWER ? tc[ax] * TS + TS > dims[ax] - R : tc[ax] == 0;
        own[ax] = wrap[ax] && tc[ax] == 0 && dims[ax] - R < TS;
    }
    // the entry of offset d along ax for the row at (x, y, z) of this tile
    auto entry = [&](int ax, int d, int x, int y, int z) -> T {
        if constexpr (!TRANS) {
            return a.F[(size_t)islot(ax, d) * m.np + tile + ((z % TS) * TS + y % TS) * TS + x % TS];
        } else {
            int c[3] = {x, y, z};
            const int n = dims[ax];
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (q == ax) {
                    c[q] += d;
                    c[q] = c[q] < 0 ? c[q] + n : (c[q] >= n ? c[q] - n : c[q]);
                }
            return a.F[(size_t)islot(ax, -d) * m.np + m.row(c[0], c[1], c[2])];
        }
    };
    // place of the row (lx, ly, lz) in fs: its index, or its rank in level
    // order within the half (rows of lower levels, then [y][x] order)
    auto place = [&](int px, int py, int pz) -> int {
        if constexpr (NCH == 1) return (pz * TS + py) * TS + px;
        // by the level's distance from the nearer corner: level L < 11 has
        // (rows below it) + (rows of it with a smaller (y, x)) before it; the
        // other half mirrors it
        const bool up = px + py + pz >= LCH;
        if (up) {
            px = TS - 1 - px;
            py = TS - 1 - py;
            pz = TS - 1 - pz;
        }
        const int L = px + py + pz;
        // rows of a level k <= 10 whose y is below y0: sum over y < y0 of the x with 0 <= k - y - x < 8
        auto upto = [](int k, int y0) {
            int t = 0;
#pragma unroll
            for (int y = 0; y < TS; y++) {
                const int e = k - y;                         // x + z
                const int cnt = e < 0 ? 0 : (e < TS ? e + 1 : 2 * TS - 1 - e);
                t += y < y0 ? cnt : 0;
            }
            return t;
        };
        int r = 0;
#pragma unroll
        for (int k = 0; k < LCH; k++) r += k < L ? upto(k, TS) : 0;
        const int e = L - py;
        return r + upto(L, py) + px - (e < TS ? 0 : e - TS + 1);
    };
    auto exists = [&](int c, int n, int d) { return LOWER ? c + d >= 0 : c + d < n; };

    // factor rows of half ch: the 18 entries towards the halo, zero where no
    // column is (its value is zero too, so the product leaves the sum as it
    // is), and 1/u_ii
    auto stage = [&](int ch) {
#pragma unroll
        for (int h = 0; h < ILU_TP / ILU_NT; h++) {
            const int e = tid + h * ILU_NT;
            const int px = e % TS, py = e / TS % TS, pz = e / (TS * TS);
            const int c[3] = {tc[0] * TS + px, tc[1] * TS + py, tc[2] * TS + pz};
            const bool here = NCH == 1 || (px + py + pz >= LCH) == (ch == 1);
            const bool ok = here && c[0] < a.nx && c[1] < a.ny && c[2] < a.nz;
            T f[NSL];
            if (NCH == 1 && !TRANS) {
                // padded rows are there to be read: no branch before the loads
#pragma unroll
                for (int ax = 0; ax < 3; ax++)
#pragma unroll
                    for (int j = 0; j < R; j++) f[ax * R + j] = a.F[(size_t)islot(ax, LOWER ? j - R : j + 1) * m.np + tile + e];
                if (DIAG) f[NSL - 1] = a.F[tile + e];
            } else if (ok) {
#pragma unroll
                for (int ax = 0; ax < 3; ax++)
#pragma unroll
                    for (int j = 0; j < R; j++) f[ax * R + j] = entry(ax, LOWER ? j - R : j + 1, c[0], c[1], c[2]);
                if (DIAG) f[NSL - 1] = a.F[tile + e];
            }
            const int q = place(px, py, pz);
            if constexpr (NCH > 1) plc[e] = (unsigned char)q;
            if (here) {
#pragma unroll
                for (int ax = 0; ax < 3; ax++)
#pragma unroll
                    for (int j = 0; j < R; j++)
                        fs[ax * R + j][q] = s_sel(ok && exists(c[ax], dims[ax], LOWER ? j - R : j + 1), f[ax * R + j], zero);
                if (DIAG) fs[NSL - 1][q] = s_sel(ok, f[NSL - 1], zero);
            }
        }
    };
    // halos, boundary values and the tile's right-hand side by lines (zero past
    // the grid and where no column is): one axis a wavefront.  Loaded before
    // the factor rows, parked after them.
    T hl[R], hw[R], hr[TS];
    const int hax = min(tid >> 6, 2);
    // (selects: a runtime index would put the arrays in scratch memory)
    auto of = [&](auto x0, auto x1, auto x2) { return hax == 0 ? x0 : (hax == 1 ? x1 : x2); };
    // fast and slow coordinate of a line
    const int g0 = of(tc[1], tc[0], tc[0]) * TS + lx, g1 = of(tc[2], tc[2], tc[1]) * TS + ly;
    const int hn = of(dims[0], dims[1], dims[2]), hc = of(tc[0], tc[1], tc[2]) * TS;
    const bool hok = g0 < of(dims[1], dims[0], dims[0]) && g1 < of(dims[2], dims[2], dims[1]);
    const bool hwrap = of(wrap[0], wrap[1], wrap[2]);
    {
        const size_t sa = of(st[0], st[1], st[2]);
        const size_t base = hok ? g0 * of(st[1], st[0], st[0]) + g1 * of(st[2], st[2], st[1]) : 0;
        auto at = [&](int col) { return base + (size_t)min(max(col, 0), hn - 1) * sa; };
#pragma unroll
        for (int j = 0; j < R; j++) {
            hl[j] = io[at(LOWER ? hc - R + j : hc + TS + j)];
            hw[j] = io[at(LOWER ? j : hn - R + j)];
        }
#pragma unroll
        for (int j = 0; j < TS; j++) hr[j] = in[at(hc + j)];
    }
    // Entries across the boundary.  With cc = c - (n - R) (below; above: R - 1 -
    // c) a row of such a line has cc + 1 of them, in ascending columns k = 0 ..
    // cc at d = R - cc + k (below: column k; above: d = k - R, column n - R + c + k).
    // Staged as products with those columns' values (in an own line, alone).
    if constexpr (WST) {
#pragma unroll
        for (int ax = 0; ax < 3; ax++)
            if (wrap[ax])
                for (int e = tid; e < TS * TS * NT3; e += ILU_NT) {
                    const int l = e % (TS * TS), t = e / (TS * TS);
                    int cc = 0;
#pragma unroll
                    for (int q = 1; q < R; q++) cc = t >= q * (q + 1) / 2 ? q : cc;
                    const int k = t - cc * (cc + 1) / 2;
                    const int c = LOWER ? dims[ax] - R + cc : R - 1 - cc;
                    const int a0 = ax == 0 ? 1 : 0, a1 = ax == 2 ? 1 : 2;
                    int g[3];
                    g[ax] = c;
                    g[a0] = tc[a0] * TS + l % TS;
                    g[a1] = tc[a1] * TS + l / TS;
                    const bool ok = c / TS == tc[ax] && g[a0] < dims[a0] && g[a1] < dims[a1];
                    T v = zero;
                    if (ok) {
                        v = entry(ax, LOWER ? R - cc + k : k - R, g[0], g[1], g[2]);
                        g[ax] = LOWER ? k : dims[ax] - R + c + k;
                        if (!own[ax]) v = s_mul(v, io[g[0] * st[0] + g[1] * st[1] + g[2] * st[2]]);
                    }
                    wf[ax][e] = v;
                }
    }
    stage(LOWER ? 0 : NCH - 1);
    if (skip) return;
    if (tid < 192) {
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int col = LOWER ? hc - R + j : hc + TS + j;
            ln[hax][lane][HB + j] = s_sel(hok && col >= 0 && col < hn, hl[j], zero);
            wr[hax][lane][j] = s_sel(hok && hwrap, hw[j], zero);
        }
#pragma unroll
        for (int j = 0; j < TS; j++) ln[hax][lane][C0 + j] = s_sel(hax == 2 && hok && hc + j < hn, hr[j], zero);
    }
    __syncthreads();

    const int x = tc[0] * TS + lx, y = tc[1] * TS + ly;
    // what a level needs besides the values of the level before it
    struct Level {
        T p[3][R];               // products (f of column J1 instead)
        T w[3][R];               // products across the boundary
        T rhs, dinv;
    };
    Level cur;
    T f[3][R], u[3][R], wfv[3][R], rhs, dinv;
    auto lz_of = [&](int s) { return LOWER ? s - lx - ly : NL - 1 - s - lx - ly; };
    // reads for level s (in bounds at any s; of use where the lane has a row)
    auto reads = [&](int s, int ch) {
        const int lz = min(max(lz_of(s), 0), TS - 1);
        const int cell[3] = {lx, ly, lz};
        const int line[3] = {lz * TS + ly, lz * TS + lx, lane};
        const int q = NCH == 1 ? lz * TS * TS + lane : plc[lz * TS * TS + lane];
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const T *l = &ln[ax][line[ax]][C0 + cell[ax] + (LOWER ? -R : 1)];
#pragma unroll
            for (int j = 0; j < R; j++) {
                f[ax][j] = fs[ax * R + j][q];
                if (j != J1) u[ax][j] = l[j];
            }
            if (wrap[ax]) {
                // (places past a row's own are read within the arrays, not used)
                const int c = tc[ax] * TS + cell[ax];
                const int cc = min(max(LOWER ? c - (dims[ax] - R) : R - 1 - c, 0), R - 1);
#pragma unroll
                for (int k = 0; k < R; k++) {
                    const int col = min(LOWER ? k : c + k, R - 1);
                    if constexpr (WST) {
                        wfv[ax][k] = wf[ax][(cc * (cc + 1) / 2 + k) * TS * TS + line[ax]];
                        if (own[ax]) wfv[ax][k] = s_mul(wfv[ax][k], wr[ax][line[ax]][col]);
                    } else {
                        wfv[ax][k] = zero;
                        if (k <= cc)
                            wfv[ax][k] = s_mul(entry(ax, LOWER ? R - cc + k : k - R, x, y, tc[2] * TS + lz),
                                               wr[ax][line[ax]][col]);
                    }
                }
            }
        }
        rhs = ln[2][lane][C0 + lz];
        if (DIAG) dinv = fs[NSL - 1][q];
    };
    auto products = [&]() {
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
#pragma unroll
            for (int j = 0; j < R; j++) cur.p[ax][j] = j == J1 ? f[ax][j] : s_mul(f[ax][j], u[ax][j]);
            if (wrap[ax]) {
#pragma unroll
                for (int k = 0; k < R; k++) cur.w[ax][k] = wfv[ax][k];
            }
        }
        cur.rhs = rhs;
        if (DIAG) cur.dinv = dinv;
    };
    auto level = [&](int s, int ch, bool more) {
        const int lz = lz_of(s);
        const int z = tc[2] * TS + lz;
        const bool live = lz >= 0 && lz < TS && x < a.nx && y < a.ny && z < a.nz;
        const int lzc = min(max(lz, 0), TS - 1);
        const int cell[3] = {lx, ly, lzc};
        const int line[3] = {lzc * TS + ly, lzc * TS + lx, lane};
        // the three values of the level before
        T u1[3];
#pragma unroll
        for (int ax = 0; ax < 3; ax++) u1[ax] = ln[ax][line[ax]][C0 + cell[ax] + (LOWER ? -1 : 1)];
        if (more) reads(s + 1, ch);
        T sum = cur.rhs;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const int ax = LOWER ? 2 - t : t;            // ascending column index
            // columns across the boundary: below the row they come first,
            // above it last
            auto across = [&]() {
                if (!wrap[ax]) return;
                const int c = tc[ax] * TS + cell[ax];
                const int cc = LOWER ? c - (dims[ax] - R) : R - 1 - c;
#pragma unroll
                for (int k = 0; k < R; k++) sum = s_sel(k <= cc, s_sub(sum, cur.w[ax][k]), sum);
            };
            if (LOWER) across();
#pragma unroll
            for (int j = 0; j < R; j++) sum = s_sub(sum, j == J1 ? s_mul(cur.p[ax][j], u1[ax]) : cur.p[ax][j]);
            if (!LOWER) across();
        }
        if (DIAG) sum = s_mul(sum, cur.dinv);
        if (live) {
            const int cr[3] = {x, y, z};
#pragma unroll
            for (int ax = 0; ax < 3; ax++) {
                ln[ax][line[ax]][C0 + cell[ax]] = sum;
                if (own[ax]) {
                    const int j = LOWER ? cr[ax] : cr[ax] - (dims[ax] - R);
                    if (j >= 0 && j < R) wr[ax][line[ax]][j] = sum;
                }
            }
            io[x * st[0] + y * st[1] + z * st[2]] = sum;
        }
        if (more) products();
        // one wavefront: orders this level's LDS writes before the next's reads
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll 1
    for (int h = 0; h < NCH; h++) {
        const int ch = LOWER ? h : NCH - 1 - h;
        if (h > 0) {
            __syncthreads();                     // the levels of the other half are done with fs
            stage(ch);
            __syncthreads();
        }
        if (tid < 64) {
            reads(h * LCH, ch);
            products();
#pragma unroll 1
            for (int s = h * LCH; s + 1 < (h + 1) * LCH; s++) level(s, ch, true);
            level((h + 1) * LCH - 1, ch, false);
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
size_t ilu_values(int nx, int ny, int nz) { return TileMap(nx, ny, nz).np * ILU_ROW; }

// the (ti, tj) box of tile diagonal D
template <typename T>
static IluArgsT<T> on_diagonal(IluArgsT<T> a, const TileMap &m, int D)
{
    a.diag_tiles = D;
    a.t0x = std::max(0, D - (m.ty - 1) - (m.tz - 1));
    a.t0y = std::max(0, D - (m.tx - 1) - (m.tz - 1));
    a.wx = std::min(m.tx - 1, D) - a.t0x + 1;
    a.wy = std::min(m.ty - 1, D) - a.t0y + 1;
    return a;
}

template <typename T>
hipError_t ilu_factor(const IluArgsT<T> &a, hipStream_t st)
{
    const TileMap m(a.nx, a.ny, a.nz);
    for (int D = 0; D < m.tx + m.ty + m.tz - 2; D++) {
        const IluArgsT<T> b = on_diagonal(a, m, D);
        const dim3 g(b.wx * b.wy), wg(64);
        if (std::min({a.nx, a.ny, a.nz}) > 3 * R) hipLaunchKernelGGL((ilu_factor_kernel<T, false>), g, wg, 0, st, b);
        else hipLaunchKernelGGL((ilu_factor_kernel<T, true>), g, wg, 0, st, b);
    }
    return hipGetLastError();
}

template <typename T>
hipError_t ilu_apply(const IluArgsT<T> &a0, const T *in, T *out, bool trans, const int *skip, hipStream_t st)
{
    IluArgsT<T> a = a0;
    a.skip = skip;
    const TileMap m(a.nx, a.ny, a.nz);
    const int nd = m.tx + m.ty + m.tz - 2;
    // forward: L (or U^T) over ascending tile diagonals, reading `in`
    for (int D = 0; D < nd; D++) {
        const IluArgsT<T> b = on_diagonal(a, m, D);
        const dim3 g(b.wx * b.wy), wg(ILU_NT);
        if (trans) hipLaunchKernelGGL((ilu_solve_kernel<T, true, true, true>), g, wg, 0, st, b, in, out);
        else hipLaunchKernelGGL((ilu_solve_kernel<T, true, false, false>), g, wg, 0, st, b, in, out);
    }
    // backward: U (or L^T) over descending ones, in place
    for (int D = nd - 1; D >= 0; D--) {
        const IluArgsT<T> b = on_diagonal(a, m, D);
        const dim3 g(b.wx * b.wy), wg(ILU_NT);
        if (trans) hipLaunchKernelGGL((ilu_solve_kernel<T, false, true, false>), g, wg, 0, st, b, (const T *)out, out);
        else hipLaunchKernelGGL((ilu_solve_kernel<T, false, false, true>), g, wg, 0, st, b, (const T *)out, out);
    }
    return hipGetLastError();
}

template hipError_t ilu_factor<double>(const IluArgsT<double> &, hipStream_t);
template hipError_t ilu_factor<double2>(const IluArgsT<double2> &, hipStream_t);
template hipError_t ilu_apply<double>(const IluArgsT<double> &, const double *, double *, bool, const int *, hipStream_t);
template hipError_t ilu_apply<double2>(const IluArgsT<double2> &, const double2 *, double2 *, bool, const int *,
                                       hipStream_t);

}  // namespace aar
