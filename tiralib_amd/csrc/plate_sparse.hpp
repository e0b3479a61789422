// plate_sparse.hpp -- the listed-voter form of the tabulated learned-plate vote.
#pragma once
#include "mlp.hpp"
#include "vote3.hpp"

namespace th {

// Offset (du, dv, dw): unit direction and attenuations (vote3.hip).
void offset_geometry(int du, int dv, int dw, float s1, float s2, float d[3], float& c1, float& c2);

// Most distinct distance rows the listed gather's LDS holds.
unsigned plate_sparse_max_rows();

// Votes the plates of the padded payload `pay` ((n, scale) per voxel of `g`)
// for the receivers of every 64 x 4 x bz tile whose voters are few, through
// the network table `vtab`; writes those receivers' votes to `out`
// (`accumulate`: adds them). *tiles: one flag per tile (x fastest, then y),
// 1 where this call votes and 0 where the window gather has to; NULL when it
// has to everywhere (no list memory, window or volume outside this form).
int plate_sparse_run(const float4* pay, const float4* vtab, int vtab_rows, float sigma1, const VoteGeom& g, int bz,
                     float* out, int layout, bool accumulate, hipStream_t st, const unsigned char** tiles);

}  // namespace th
