// ilu.h -- ILU(0) of the periodic FD12 star matrix, real and complex (see
// ilu.hip).
#pragma once

#include "aar_common.h"

namespace aar {

constexpr int ILU_ROW = 37;          // values of a row: 1/u_ii and the 36 off-diagonals
constexpr int ILU_TS = 8;            // tile side
constexpr int ILU_TP = ILU_TS * ILU_TS * ILU_TS;

template <typename T>
struct IluArgsT {
    int nx, ny, nz;
    int diag_tiles;              // the tile diagonal ti + tj + tk of this launch
    int t0x, t0y, wx, wy;        // its (ti, tj) box
    double w[R + 1];             // a * coeff[o]
    double diag;                 // real part of the diagonal without c(x): a * 3 * coeff[0] (+ sigma, + c0)
    double eta;                  // its imaginary part (complex matrix)
    const double *c;             // + c(x) on the diagonal, or null
    T *F;                        // ilu_values(nx, ny, nz) values
    const int *skip;             // nonzero: no work (solver stopped / step gated)
};
using IluArgs = IluArgsT<double>;

// values held by the factors of a grid
size_t ilu_values(int nx, int ny, int nz);
// every side >= 13
template <typename T>
hipError_t ilu_factor(const IluArgsT<T> &a, hipStream_t st);
// out = M^{-1} in (trans: M^{-T} in); out may be in
template <typename T>
hipError_t ilu_apply(const IluArgsT<T> &a, const T *in, T *out, bool trans, const int *skip, hipStream_t st);

}  // namespace aar
