// Nonlocal projector steps on the matrix cores (kernels_nonlocal.hip), for
// atoms of at most kTileAtomPts sphere points.
#pragma once

#include "kernels.hpp"

namespace lynx {
namespace gpu {

constexpr int kTileAtomPts = 1024;

// What one launch does for each (atom, column): the gather beta_out =
// dV Gamma chi^T y, or the scatter y += a chi beta_in and then the gather of
// the result.  An update needs spheres that share no grid point
// (NlDev::disjoint).  A scatter alone stays with nl_scatter, whose lanes run
// over all covered points in memory order (216 atoms x 480 columns of 90^3
// float: 188 us against 250 us by tiles).
enum NlMode { kNlGather = 1, kNlUpdate = 2 };

bool nl_tile_fits(const NlDev &nl, NlMode mode);
// y is read only in a gather; with acoef (device memory, arithmetic type) a
// is read from acoef[0].
void nl_tile(int e, const NlDev &nl, NlMode mode, const void *beta_in, void *beta_out, void *y, long ldy, int ncol,
             double a, hipStream_t st, const void *acoef = nullptr);

// Batched: work items of a unit are its n_atom x nl_tile_groups(e, ncol)
// (atom, column group) pairs, atoms fastest; recs are the batch's records.
int nl_tile_groups(int e, int ncol);
int nl_tile_waves(int max_atom_pts);
void nl_tile_batch(int e, int npm, const void *recs, const int *items, int nitems, int waves, NlMode mode,
                   const void *beta_in, void *beta_out, const void *coef, int iy, hipStream_t st);

}  // namespace gpu
}  // namespace lynx
