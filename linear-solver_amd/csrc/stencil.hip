// stencil.hip -- the FD12 (radius-6, 37-point) periodic star stencil and
// the kernels that fuse it with the solver sweeps around it.
//
// Reference operator: MPI_REAL/system.c:189-205 (1-rank branch of
// Lap_Vec_mult): y = (x*3)*w0; for o = 1..6:
//   y += (x[i-o] + x[i+o] + x[j-o] + x[j+o] + x[k-o] + x[k+o]) * w_o,
// w_o = a*coeff_lap[o].  The same operation order is used here with
// contraction off, so a stencil result is bit-identical to the reference.
//
// Two forms of the sweep share the point formulas (stencil_point.h):
//
// The march (stencil_body.h), for grids that fill the chip: a block of WY
// wavefronts owns a column of 64 (narrow grids 32 or 16: march_width) x TY
// points over a z-chunk of `lz` planes
// and marches it in z.
// * z-neighbours come from a per-thread register queue of 13 planes, so
//   every plane of the column is read from HBM once per chunk;
// * x/y-neighbours come from a double-buffered LDS tile of the current
//   plane with a 6-wide halo (corners are not needed by a star stencil),
//   one barrier per plane; halo vectors are fetched R planes ahead, together
//   with the queue plane, and parked in an LDS ring;
// * block ids are mapped XCD-aware onto tiles so that y-adjacent tiles
//   (whose halos overlap) run on the same XCD and share its L2.
// What bounds it: with one point a lane the plane tile was read 8 (FP32: 4)
// bytes a lane, 21 values a point, and the LDS pipe took 1.5 of the 2.2
// clocks per point and CU at 512^3 FP64.  With 16 bytes a lane (Lane in
// stencil_point.h) it takes 0.7, and HBM bounds the sweep.  Recurrence sweep
// at 512^3: FP64 487 -> 436 us (4.9 TB/s of the two vectors), FP32 285 -> 230
// us; the true residual 680 -> 580 us.
//
// Rows that are no multiple of 16 bytes keep 16-byte accesses (x_mode).
//
// The one-shot boxes (stencil_tile.h), for the smaller grids.
//
// The epilogue of each mode fuses the pointwise work of the solver step
// that consumes A*x, so that step costs one pass over the grid.
#include "stencil_launch.h"

#include <algorithm>

namespace aar {

// ---------------------------------------------------------------------------
// host-side launch
// ---------------------------------------------------------------------------

// Rows of a one-shot box: four wavefronts, one vector per thread.
template <typename T> static int tile_rows(int lz) { return 256 * Lane<T>::V / tile_x<T>(lz); }

// 64, but where rows are no multiple of a vector and too narrow for tiles of 64
// that start early (XSHIFT) the widest of 32 and 16 that leaves room for them.
// FP32 operator, 64 wide point by point / this: 65 x 600 x 500 136 / 88 us, 61 wide
// 80 / 64, 37 wide 74 / 59, 29 wide 72 / 47.  FP64 loses less by points (8 bytes
// each), so only where fewer lanes are left idle: 65 wide 165 / 127, 29 wide 86 /
// 66, but an AAR iteration at 45 wide (32 as idle as 64) 144 / 155 and at 37 (16) 130 /
// 141.
template <typename T>
int march_width(int nx, int ny)
{
    auto lanes = [&](int w) { return (nx + w - 1) / w * w; };
    if (x_mode<T>(nx, ny, TX) != XPOINT) return TX;
    for (int w : {32, 16})
        if (x_mode<T>(nx, ny, w) == XSHIFT && (sizeof(T) == 4 || 4 * lanes(w) <= (w == 32 ? 3 : 2) * lanes(TX))) return w;
    return TX;
}

// Where the boxes are faster than the march (microseconds, march / boxes, nx a
// multiple of 4 and one more):
//                   recurrence                   true residual  PGR step
//   FP64 114^3      34.1 / 16.6   34.2 / 16.9    40.7 / 17.8    41.6 / 18.4
//        160^3      35.0 / 25.8   36.3 / 30.6    40.9 / 29.2    43.4 / 31.2
//        200x161x150 37.4 / 35.3                 43.6 / 40.0    47.7 / 44.4
//        172x171x171 38.0 / 34.7  (171) 38.5 / 35.4  44.5 / 41.5  48.1 / 44.2
//        182^3      38.3 / 40.1   38.1 / 40.9    47.3 / 48.9    49.8 / 55.1
//        192^3      39.8 / 44.5   44.1 / 48.7    47.5 / 50.9    51.0 / 56.7
//        204x203x204 47.7 / 55.7  48.9 / 56.6    60.4 / 66.3    67.3 / 76.2
//   FP32 160^3      22.9 / 17.2   24.1 / 18.2
//        192^3      25.1 / 22.5   28.8 / 26.5
//        204x203x204 31.8 / 28.9  32.4 / 29.1
// The operator alone, CG's sweeps and the ones with c(x) cross at the same
// sizes: FP64 between 5.5 and 6.0 million points (CG at 176^3, 5.5 million, 99 us an
// iteration with the boxes, 103 with the march), FP32 above 8.4 million (256^3,
// sweep alone, 41 / 50).  FP64 grids whose sides leave more than a quarter more
// of the march's 64 x 32 columns idle than of the 32 x 16 boxes keep the boxes
// up to there (recurrence: 1.33 times the lanes 300 x 40 x 520 43.6 / 40.3, 80 x
// 300 x 300 49.7 / 43.1, twice 28 x 500 x 500 56.7 / 40.5; 1.28 times 130 x 230 x
// 230 47.6 / 46.2; 1.2 times 160 x 214 x 214 41.6 / 44.9).  FP32 boxes that go point
// by point (x_mode) give way to the march in narrow columns earlier: from 2.4
// million lanes of their 64-wide tiles (61 x 200 x 200, 2.6 million lanes, 20.5 /
// 22.4; 65 x 140 x 140, 2.5, 20.5 / 22.2; 61 x 140 x 140, 1.3, 20.1 / 17.3), from 4.5
// million against columns of 16 (25 x 200 x 200, 2.6, 22.8 / 16.5; 37 x 300 x 300,
// 5.8, 26.6 / 28.6).  Boxes of 4 planes read (4 + 12)/4
// values a point; while they are about one a CU or fewer, boxes of 2 planes are
// shorter (FP32 96^3 8.7 -> 8.3 us, FP64 true residual 64^3 7.9 -> 6.2; 128^3
// 15.8 -> 16.8), and of one plane while those leave half the CUs idle (48^3
// 5.2 -> 4.9, FP32 4.9 -> 4.4, 16^3 4.9 -> 4.0; FP64 64^3 8.2 -> 8.5).  32-bit
// offsets span the grid.
template <typename T>
int stencil_tile_planes(int nx, int ny, int nz)
{
    const long n = (long)nx * ny * nz;
    if (n > 8500000L) return 0;
    auto lanes = [&](int w, int rows) { return (long)((nx + w - 1) / w * w) * ((ny + rows - 1) / rows * rows); };
    const int mw = march_width<T>(nx, ny);
    const bool idle = 4 * lanes(mw, narrow_rows<T>() * TX / mw) > 5 * lanes(tile_x<T>(4), tile_rows<T>(4));
    if (sizeof(T) == 8 && !idle && n > 5600000L) return 0;
    if (sizeof(T) == 4 && mw < TX && lanes(TX, 1) * nz > (mw == 32 ? 2400000L : 4500000L)) return 0;
    auto cols = [&](int lz) {
        return (long)((nx + tile_x<T>(lz) - 1) / tile_x<T>(lz)) * ((ny + tile_rows<T>(lz) - 1) / tile_rows<T>(lz));
    };
    if (cols(1) * ((nz + 1) / 2) <= 150) return 1;
    return cols(4) * ((nz + 3) / 4) <= 300 ? 2 : 4;
}

template <typename T>
void stencil_geometry(SArgs<T> &a, const Shape &sh)
{
    int tx = sh.w, ty = sh.wy * sh.py;
    if (wide_plane<T>(a.nx, a.ny)) ty = WIDE_ROWS;
    else if (sh.tile) tx = tile_x<T>(sh.tile), ty = tile_rows<T>(sh.tile);
    else if (sh.w < TX) ty = narrow_rows<T>() * TX / sh.w;
    a.nxy = a.nx * a.ny;
    a.ntx = (a.nx + tx - 1) / tx;
    a.nty = (a.ny + ty - 1) / ty;
    if (sh.tile) {
        a.lz = sh.tile;
    } else {
        if (a.lz <= 0) a.lz = a.nz;
        if (a.lz > a.nz) a.lz = a.nz;
    }
    a.nzc = (a.nz + a.lz - 1) / a.lz;
    a.nitems = a.ntx * a.nty * a.nzc;
}

template <typename T>
hipError_t launch_stencil(SMode m, const SArgs<T> &a, const Shape &sh, hipStream_t st)
{
    if (a.vf) return launch_stencil_vc<T>(m, a, sh, st);
    switch (m) {
    case SMode::MATVEC: return launch_sweep<T, SMode::MATVEC, false>(a, sh, st);
    case SMode::AAR_TRUE: return launch_sweep<T, SMode::AAR_TRUE, false>(a, sh, st);
    case SMode::AAR_REC: return launch_sweep<T, SMode::AAR_REC, false>(a, sh, st);
    default: break;
    }
    if constexpr (sizeof(T) == 8) {              // the FP64 solvers' own sweeps
        switch (m) {
        case SMode::RESID: return launch_sweep<T, SMode::RESID, false>(a, sh, st);
        case SMode::PGR_STEP: return launch_sweep<T, SMode::PGR_STEP, false>(a, sh, st);
        case SMode::CG_Q: return launch_sweep<T, SMode::CG_Q, false>(a, sh, st);
        case SMode::CG_RESID: return launch_sweep<T, SMode::CG_RESID, false>(a, sh, st);
        default: break;
        }
    }
    return hipErrorInvalidValue;
}

template <typename T>
int stencil_items(const SArgs<T> &a0, const Shape &sh)
{
    SArgs<T> a = a0;
    stencil_geometry(a, sh);
    return a.nitems;
}

template hipError_t launch_stencil<double>(SMode, const SArgs<double> &, const Shape &, hipStream_t);
template hipError_t launch_stencil<float>(SMode, const SArgs<float> &, const Shape &, hipStream_t);
template int stencil_items<double>(const SArgs<double> &, const Shape &);
template int stencil_items<float>(const SArgs<float> &, const Shape &);
template void stencil_geometry<double>(SArgs<double> &, const Shape &);
template void stencil_geometry<float>(SArgs<float> &, const Shape &);
template int march_width<double>(int, int);
template int march_width<float>(int, int);
template int stencil_tile_planes<double>(int, int, int);
template int stencil_tile_planes<float>(int, int, int);

}  // namespace aar
