// Launches of the one-point-per-thread stencil step (stencil_points.hpp),
// one translation unit per element type.
#pragma once

#include "kernels.hpp"

namespace lynx {
namespace gpu {

// Launch shape: band rows per workgroup, threads, halo points per thread, LDS
// row pitch, z-chunks, whether the whole z range is marched once, LDS bytes.
struct PointShape {
    int tyr = 0, nt = 0, hp = 0, pitch = 0, nzch = 1;
    bool wrapz = false;
    size_t lds = 0;
};

// Shape for element type e with at most max_threads threads (64..512) and
// nzch z-chunks; false when the rows do not fit.
bool point_shape(int e, const StencilGeom &g, int max_threads, int nzch, PointShape &out);
// Shape for a unit of a batch (one z-chunk).
bool point_shape_batch(int e, const StencilGeom &g, PointShape &out);

void points_step(int e, const StencilGeom &g, const void *x, long ldx, const void *old, long ldo, void *out,
                 long ldout, const void *veff, int ncol, double a, double b, double s, const PointShape &sh,
                 hipStream_t st, const void *coef);
// recs: the batch's device records (BatchRec of e's arithmetic type)
void points_batch(int e, const void *recs, const int *items, int nitems, bool nonorth, const void *coef, int ix,
                  int iold, int iout, const PointShape &sh, hipStream_t st);

#define LYNX_POINTS_DECLARE(tag)                                                                                \
    void points_step_##tag(const StencilGeom &g, const void *x, long ldx, const void *old, long ldo, void *out, \
                           long ldout, const void *veff, int ncol, double a, double b, double s,                \
                           const PointShape &sh, hipStream_t st, const void *coef);                             \
    void points_batch_##tag(const void *recs, const int *items, int nitems, bool nonorth, const void *coef,     \
                            int ix, int iold, int iout, const PointShape &sh, hipStream_t st);
LYNX_POINTS_DECLARE(f64)
LYNX_POINTS_DECLARE(c128)
LYNX_POINTS_DECLARE(f32)
LYNX_POINTS_DECLARE(c64)
#undef LYNX_POINTS_DECLARE

}  // namespace gpu
}  // namespace lynx
