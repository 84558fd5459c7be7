// Launch shapes and element-type dispatch of the one-point-per-thread stencil
// step.
#include "kernels_points.hpp"
#include "common.hpp"

#include <algorithm>

namespace lynx {
namespace gpu {

namespace {
constexpr long kLds = 160 * 1024;   // LDS of a workgroup (gfx950)

int round64(int n) { return (n + 63) / 64 * 64; }

// complex128 kernels with six halo points per thread hold more than a thread's
// registers, but for the orthogonal one that marches beyond the z boundary
bool spills(int e, bool orth, const PointShape &s) { return e == C128 && s.hp == 6 && (!orth || s.wrapz); }

// Whether a march that wraps in z (nz planes instead of nz + 2R) is worth the
// LDS of its end planes' parts: the workgroups left on a CU must hide each
// other's latency.  Without / with it, us for six steps of a batch by waves
// per CU: double 60^3 x 108 orthogonal 8 waves 1337 / 1423, 9 waves 1483 /
// 1413, 40^3 x 370 12 waves 1333 / 1220; complex64 72^3 8 waves 807 / 904;
// complex128 40^3 4 waves 1115 / 1345, skew 60^3 4 waves 1648 / 1949 and 48^3
// 6 waves 1825 / 1537; double skew 8 waves 1833 / 1876 (256 threads), 2259 /
// 2069 (512).
bool wrap_pays(int e, bool orth, PointShape s, long lds)
{
    s.wrapz = true;
    const int waves = (int)(kLds / lds) * (s.nt / 64);
    return waves > (orth && e != C128 ? 8 : 4) && !spills(e, orth, s);
}
}  // namespace

bool point_shape(int e, const StencilGeom &g, int max_threads, int nzch, PointShape &out)
{
    const int R = kMaxR, nx = g.nx, ny = g.ny;
    const long es = (long)elem_size(e);
    PointShape s;
    // pitches, and the halo points per thread that each one's kernels are
    // built for.  76 is for rows of 53 to 64 points, which a pitch of 128 left
    // with two workgroups of double on a CU instead of three: batches of
    // 64^3 x 91 double 1384 -> 1181 us for six steps, 60^3 x 320 3321 -> 3093 us,
    // complex64 skew 60^3 x 160 2597 -> 2205 us; alone 59^3 x 174 double 6439 ->
    // 5743 us for 20
    constexpr int pitches[5] = {40, 64, 76, 128, 256};
    constexpr int slots[5][3] = {{1, 2, 2}, {2, 3, 3}, {2, 3, 3}, {2, 3, 6}, {6, 6, 6}};
    int ip = 0;
    while (ip < 4 && nx + 2 * R > pitches[ip]) ++ip;
    s.pitch = pitches[ip];
    const int *hs = slots[ip];
    if (nx + 2 * R > 256 || nx > max_threads) return false;
    s.nzch = std::max(1, std::min(nzch, g.nz));
    for (int most = std::min(ny, max_threads / nx); most >= 1; --most) {
        const int nb = (ny + most - 1) / most;
        s.tyr = (ny + nb - 1) / nb;
        s.nt = round64(std::max(s.tyr * nx, (2 * R * nx + hs[2] - 1) / hs[2]));
        if (s.nt > 512) continue;
        s.hp = hs[2];
        for (int k = 2; k >= 0; --k)
            if (2 * R * nx <= hs[k] * s.nt) s.hp = hs[k];
        const long planes = 2 * es * s.pitch * ((s.tyr + 2 * R) + (g.orth ? 0 : s.tyr));
        const long stash = 2 * R * es * s.nt;
        s.wrapz = s.nzch == 1 && g.nz >= 2 * R && planes + stash <= kLds && wrap_pays(e, g.orth, s, planes + stash);
        s.lds = (size_t)(planes + (s.wrapz ? stash : 0));
        if (planes > kLds) continue;
        out = s;
        return true;
    }
    return false;
}

// The cost of a shape per point: idle lanes, halo rows (a tenth of an own
// row's cost each) and, with 512 threads, fewer workgroups to a CU to hide
// each other's barriers; 320 to 448 threads leave too many wave slots empty.
// Measured (rows / threads): 24^3 x 1344 complex64 skew 8/192 176 us, 12/320
// 249, 4/128 218; 32^3 x 400 8/256 136, 4/128 160, 16/512 189; double 30^3 x
// 1600 6/192 281, 8/256 289, 10/320 354, 15/512 312; 40^3 x 600 6/256 247,
// 4/192 270, 8/320 288; 50^3 x 300 5/256 246, 10/512 234, 7/384 314; 100 x 60
// x 60 x 60 5/512 191, 2/256 218, 3/320 250.
bool point_shape_batch(int e, const StencilGeom &g, PointShape &out)
{
    double best = 0;
    for (int budget : {128, 192, 256, 512}) {
        PointShape s;
        if (!point_shape(e, g, budget, 1, s)) continue;
        if (spills(e, g.orth, s) && budget < 512) continue;
        const int nb = (g.ny + s.tyr - 1) / s.tyr;
        double cost = (double)nb * s.nt / ((double)g.nx * g.ny) * (1.0 + 0.12 * 2 * kMaxR / s.tyr);
        if (s.nt > 256) cost *= 1.64;
        if (best == 0 || cost < best) {
            best = cost;
            out = s;
        }
    }
    return best > 0;
}

void points_step(int e, const StencilGeom &g, const void *x, long ldx, const void *old, long ldo, void *out,
                 long ldout, const void *veff, int ncol, double a, double b, double s, const PointShape &sh,
                 hipStream_t st, const void *coef)
{
    auto f = e == F64 ? points_step_f64 : e == C128 ? points_step_c128 : e == F32 ? points_step_f32 : points_step_c64;
    f(g, x, ldx, old, ldo, out, ldout, veff, ncol, a, b, s, sh, st, coef);
}

void points_batch(int e, const void *recs, const int *items, int nitems, bool nonorth, const void *coef, int ix,
                  int iold, int iout, const PointShape &sh, hipStream_t st)
{
    auto f = e == F64   ? points_batch_f64
             : e == C128 ? points_batch_c128
             : e == F32  ? points_batch_f32
                         : points_batch_c64;
    f(recs, items, nitems, nonorth, coef, ix, iold, iout, sh, st);
}

}  // namespace gpu
}  // namespace lynx
