// plate_sparse.hpp -- the listed-voter form of the tabulated learned-plate vote.
#pragma once
#include "mlp.hpp"
#include "vote3.hpp"

namespace th {

// Offset (du, dv, dw): unit direction and attenuations (vote3.hip).
void offset_geometry(int du, int dv, int dw, float s1, float s2, float d[3], float& c1, float& c2);

// Most distinct distance rows the listed gather's LDS holds.
unsigned plate_sparse_max_rows();

// The listed voters of a field and the tiles they serve (device).
struct PlateList {
    float4* lv = nullptr;
    uint2* lp = nullptr;
    unsigned *cnt = nullptr, *tot = nullptr, *next = nullptr;
    unsigned char* sparse = nullptr;  // per 64 x 4 x bz tile (x fastest, then y): 1 where the list votes, 0 the window gather
    float4* ent = nullptr;
    int *entrow = nullptr, *rows = nullptr, nrows = 0;
};

// Lists the voters of the padded payload `pay` ((n, scale) per voxel of `g`) and
// flags the tiles whose voters are few. *ok: false where the window gather has
// to vote everywhere (no list memory, window or volume outside this form). dense
// (optional, device): the tiles it has to vote are added to it.
int plate_list_build(const float4* pay, int vtab_rows, float sigma1, const VoteGeom& g, int bz, unsigned* dense,
                     hipStream_t st, PlateList* list, bool* ok);

// Votes the listed plates for the receivers of the flagged tiles through the
// network table `vtab` and writes them to `out` (`accumulate`: adds them). stop
// (optional, device): nothing is done where it is set.
int plate_sparse_gather(const PlateList& list, const float4* vtab, const VoteGeom& g, int bz, float* out, int layout,
                        bool accumulate, const unsigned long long* stop, hipStream_t st);

}  // namespace th
