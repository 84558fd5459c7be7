// Every LDS read of a stencil lane, with points of its own or not, lies in its
// plane, and every run has one owner: the lane map of the kernels over the
// launch shapes that their rules form.
#include "stencil_lanes.hpp"

#include <algorithm>
#include <cstdio>
#include <vector>

using namespace lynx::gpu;
constexpr int R = 6;
static long checked = 0, bad = 0;

static void inside(int at, int n, int elems)
{
    ++checked;
    if (at < 0 || at + n > elems) ++bad;
}

// run-vector kernels: x reads of every run, y reads of the first one's column
static void runs_of(int nx, int ny, int nt, int RV, int VW, bool align)
{
    const int XO = (R + VW - 1) / VW * VW, runs = nx / VW, lpr = align ? (runs + 15) / 16 * 16 : runs;
    const int rpb = nt / lpr * RV, W = nx + 2 * XO <= 64 ? 64 : 128;
    if (nx % VW || rpb < 1 || nx + 2 * XO > 128 || nx < 2 * XO) return;
    const int nb = (ny + rpb - 1) / rpb, tyr = (ny + nb - 1) / nb, elems = plane_elems(W, R, tyr, nt, VW);
    for (int y0 = 0; y0 < ny; y0 += tyr) {
        const int rows = std::min(tyr, ny - y0);
        std::vector<int> owners(rows * runs, 0);
        for (int tid = 0; tid < nt; ++tid)
            for (int r = 0; r < RV; ++r) {
                const RunLane q = run_lane(tid, r, RV, lpr, runs, rows, VW);
                const int at = plane_at(W, R, XO, q.y, q.x);
                // a run of the band, or of the row above it
                if (q.x < 0 || q.x + VW > nx || q.y < 0 || q.y > rows || (q.own && q.y == rows)) ++bad;
                else if (q.own) ++owners[q.y * runs + q.x / VW];
                inside(at - XO, 2 * XO + VW, elems);
                if (r == 0) {
                    inside(at - R * W, VW, elems);
                    inside(at + (RV - 1 + R) * W, VW, elems);
                } else if (at != plane_at(W, R, XO, run_lane(tid, 0, RV, lpr, runs, rows, VW).y + r, q.x)) ++bad;
            }
        for (int n : owners) bad += n != 1;
    }
}

// one point per slot, RP slots per thread (long rows)
static void points_of(int nx, int ny, int nt, int RP)
{
    const int W = 256, pts = nt * RP;
    if (nx > pts) return;
    int nb = std::max(1, std::min((nx * ny + pts - 1) / pts, ny)), tyr = (ny + nb - 1) / nb;
    while (tyr * nx > pts) tyr = (ny + ++nb - 1) / nb;
    const int elems = plane_elems(W, R, tyr, nt, 1);
    for (int y0 = 0; y0 < ny; y0 += tyr)
        for (int q = 0; q < pts; ++q) {
            const int npts = std::min(tyr, ny - y0) * nx, p = band_point(q, npts);
            if (p < 0 || p >= npts || (q < npts && p != q)) ++bad;
            const int at = plane_at(W, R, R, p / nx, p % nx);
            inside(at - R, 2 * R + 1, elems);
            inside(at - R * W, 1, elems);
            inside(at + R * W, 1, elems);
        }
}

int main()
{
    for (int nx = 12; nx <= 116; nx += 2)
        for (int ny : {12, 13, 30, 61})
            for (int nt : {256, 512})
                for (int rv : {1, 2})
                    for (int vw : {2, 4})
                        for (bool al : {false, true}) runs_of(nx, ny, nt, rv, vw, al);
    for (int nx : {117, 120, 200, 244})
        for (int ny : {12, 13, 40})
            for (int rp : {1, 2, 4, 8}) points_of(nx, ny, 512, rp);
    std::printf("%ld reads, %ld faults\n", checked, bad);
    return bad != 0;
}
