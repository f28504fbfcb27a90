// history.h -- helpers shared by the history kernels (Gram, update).
#pragma once

#include "aar_common.h"
#include "aar_device.h"
#include "aar_kernels.h"

namespace aar {

template <typename T> struct Vec2;
template <> struct Vec2<double> { using type = double2; };
template <> struct Vec2<float> { using type = float2; };

// reference column index of the difference column of age k (AAR.c:97,
// PGR.c:105); identity in DIRECT mode
__device__ inline int ref_col(int it, int k, int m, int direct)
{
    return direct ? k : ((it - 2 - k) % m + m) % m;
}

}  // namespace aar
