// Host rules that choose the 3D kernels' forms from a geometry (host code
// only: no device code or launch).
#pragma once

#include "internal.hpp"

namespace amx {

// Column FP (fp3d_cols.hip): rays per lane for a direction group, 0: the gather
int fp3d_cols_rays(const Geom3D &g, int grp);

struct FPForms {
    int rays[3] = {0, 0, 0};  // per direction group, as fp3d_cols_rays
    bool cols = false, gather = false;
    size_t bytes = 0;  // the volume copies' scratch
};
FPForms fp3d_forms(const Geom3D &g, unsigned ss);

// Its transpose (adj3d_cols.hip)
bool adj3d_cols_ok(const Geom3D &g, int grp);

// The matched BP's forms and scratch bytes
struct MatchedForms {
    bool cols[3] = {false, false, false};  // per direction group: split, else gather
    unsigned chunk[3] = {0, 0, 0};         // angles per pass
    size_t tables = 0, geo = 0, sums = 0;
};
MatchedForms matched_forms(const Geom3D &g, unsigned ss);

// Workgroups of the BP's 16 x 16 column kernels with 16 z voxels per thread.
// Below 1024 (4 per CU) the chip is not full: bp3d_split_kernel.
inline size_t bp3d_blocks(const Geom3D &g) {
    return (size_t)((g.nx + 15) / 16) * ((g.ny + 15) / 16) * ((g.nz + 15) / 16);
}
constexpr size_t kBpFullBlocks = 1024;

// Whether the BP's detector footprints fit the staged tiles (bp3d_tile.hip)
bool bp3d_tiles_fit(const Geom3D &g);

// Flat parallel BP (bp3d_flat.hip)
bool bp3d_flat_ok(const Geom3D &g);

}  // namespace amx
