// Where the lanes of the stencil kernels with several points per thread write
// and read a plane in LDS.  Plain constexpr functions, for the kernels and for
// host checks of their ranges.
#pragma once

namespace lynx {
namespace gpu {

// Elements of one plane buffer: W elements a row, tyr band rows with R rows
// below and above, then VW elements per thread that take the writes of points
// without a ghost copy.
constexpr int plane_elems(int W, int R, int tyr, int nt, int vw) { return W * (tyr + 2 * R) + nt * vw; }

// Element of band row y (0 is the first own row) at x; XO ghost columns.
constexpr int plane_at(int W, int R, int XO, int y, int x) { return (y + R) * W + XO + x; }

// Run r (of RV) of lane tid: band row and x of its first point.  Lane q takes
// run q % lpr of the RV adjacent rows from RV (q / lpr) on.  A lane without a
// run of its own repeats one of the last rows, so that all it reads lies in
// the plane and what it writes is what the run's owner writes; the second run
// over an odd last row is the row above the band, one of its halo rows.
struct RunLane {
    bool own;
    int y, x;
};
constexpr RunLane run_lane(int tid, int r, int RV, int lpr, int runs, int rows, int VW)
{
    const int q = tid / lpr, i = tid - q * lpr, last = (rows - 1) / RV;
    return {q <= last && i < runs && RV * q + r < rows, RV * (q < last ? q : last) + r, (i < runs ? i : runs - 1) * VW};
}

// Point q of a band of npts: slots beyond it repeat its points.
constexpr int band_point(int q, int npts) { return q < npts ? q : q % npts; }

}  // namespace gpu
}  // namespace lynx
