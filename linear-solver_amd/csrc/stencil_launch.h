// stencil_launch.h -- host-side launch of one stencil sweep in a given shape.
#pragma once

#include "stencil_body.h"
#include "stencil_tile.h"

namespace aar {

// A column of 64 x (wy*py) points (TW x (wy*py*64/TW) on narrow grids).  A
// wavefront covers RPW rows of the tile
// (2 in FP64, 4 in FP32), so wy*py rows are wy wavefronts with wy*py/(RPW wy)
// rows per thread, or fewer wavefronts where that is below one row.
template <typename T, SMode M, bool VC, int WY, int ROWS, int XM, int TW = TX>
hipError_t launch_march_x(const SArgs<T> &a, hipStream_t st)
{
    constexpr int RPW = Lane<T>::RPW;
    constexpr int W = WY * RPW <= ROWS ? WY : ROWS / RPW;
    constexpr int PY = ROWS / (W * RPW);
    static_assert(W * RPW * PY == ROWS, "whole rows");
    hipLaunchKernelGGL((stencil_kernel<T, W, PY, M, VC, XM, TW>), dim3(a.nitems), dim3(64 * W), 0, st, a);
    return hipGetLastError();
}
template <typename T, SMode M, bool VC, int WY, int ROWS>
hipError_t launch_march(const SArgs<T> &a, hipStream_t st)
{
    switch (x_mode<T>(a.nx, a.ny, TX)) {
    case XVEC: return launch_march_x<T, M, VC, WY, ROWS, XVEC>(a, st);
    case XSHIFT: return launch_march_x<T, M, VC, WY, ROWS, XSHIFT>(a, st);
    default: return launch_march_x<T, M, VC, WY, ROWS, XPOINT>(a, st);
    }
}

template <typename T, SMode M, bool VC, int LZ>
hipError_t launch_boxes(const SArgs<T> &a, hipStream_t st)
{
    const dim3 grid(a.nitems), block(256);
    switch (x_mode<T>(a.nx, a.ny, tile_x<T>(LZ))) {
    case XVEC: hipLaunchKernelGGL((stencil_tile_kernel<T, 4, 1, LZ, M, VC, XVEC>), grid, block, 0, st, a); break;
    case XSHIFT: hipLaunchKernelGGL((stencil_tile_kernel<T, 4, 1, LZ, M, VC, XSHIFT>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((stencil_tile_kernel<T, 4, 1, LZ, M, VC, XPOINT>), grid, block, 0, st, a); break;
    }
    return hipGetLastError();
}

template <typename T, SMode M, bool VC>
hipError_t launch_sweep(SArgs<T> a, const Shape &sh, hipStream_t st)
{
    stencil_geometry(a, sh);
    if (wide_plane<T>(a.nx, a.ny)) return launch_march_x<T, M, VC, 8, WIDE_ROWS, XWIDE>(a, st);
    // narrow grids: one launch shape, the default one's wavefronts and rows
    constexpr int NWY = sizeof(T) == 8 ? 8 : 4;
    if (sh.tile == 0 && sh.w == 32) return launch_march_x<T, M, VC, NWY, narrow_rows<T>(), XSHIFT, 32>(a, st);
    if (sh.tile == 0 && sh.w == 16) return launch_march_x<T, M, VC, NWY, narrow_rows<T>(), XSHIFT, 16>(a, st);
    switch (sh.tile) {
    case 0: break;
    case 1: return launch_boxes<T, M, VC, 1>(a, st);
    case 2: return launch_boxes<T, M, VC, 2>(a, st);
    case 4: return launch_boxes<T, M, VC, 4>(a, st);
    default: return hipErrorInvalidValue;
    }
    switch (sh.wy * 10 + sh.py) {
    case 42: return launch_march<T, M, VC, 4, 8>(a, st);
    case 44: return launch_march<T, M, VC, 4, 16>(a, st);
    case 82: return launch_march<T, M, VC, 8, 16>(a, st);
    case 84: return launch_march<T, M, VC, 8, 32>(a, st);
    case 48: return launch_march<T, M, VC, 4, 32>(a, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace aar
