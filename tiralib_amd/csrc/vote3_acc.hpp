// vote3_acc.hpp -- the receiver accumulator of the 3D vote gathers and its
// output, shared by the window gathers (vote3.hip) and the listed-voter plate
// gather (plate_sparse.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "tira_hip.h"

namespace th {

// Sum of a receiver's votes: the six components and the isotropic part.
struct Acc {
    float xx, xy, xz, yy, yz, zz, ii;
};

__device__ __forceinline__ void write_out(float* __restrict__ out, int layout, size_t v, const Acc& a,
                                          bool add = false) {
    const float xx = a.xx + a.ii, yy = a.yy + a.ii, zz = a.zz + a.ii;
    if (layout == TIRA_LAYOUT_MAT9) {
        float* o = out + v * 9;
        const float t[9] = {xx, a.xy, a.xz, a.xy, yy, a.yz, a.xz, a.yz, zz};
        for (int k = 0; k < 9; k++) o[k] = add ? o[k] + t[k] : t[k];
    } else {
        float* o = out + v * 6;
        const float t[6] = {xx, a.xy, a.xz, yy, a.yz, zz};
        for (int k = 0; k < 6; k++) o[k] = add ? o[k] + t[k] : t[k];
    }
}

}  // namespace th
