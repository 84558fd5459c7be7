// Fused stencil step of any element type and cell with one point per thread
// and the z-terms accumulated forward, and its launches.  Included by the HIP
// sources that instantiate it, one per element type.
#pragma once

#include "kernels_points.hpp"
#include "stencil_common.hpp"

#include <algorithm>

namespace lynx {
namespace gpu {
namespace {

// Loads of one plane, issued a plane ahead of their use.
template <class S, int HP>
struct PointLoads {
    S front;                    // the owned point of the plane
    S old;                      // Y_{k-2} of the output plane
    typename Tr<S>::A v;        // Veff of the plane
    S halo[HP];                 // halo rows of the plane
};

// One workgroup owns a band of full x rows of one column and marches along z;
// a thread owns one point of the band.  Each plane passes through LDS once,
// as the newest plane f: its in-plane terms go to output f, its z-terms to
// the 2R outputs within R of it (2R+1 accumulators, as many registers as a
// ring of planes), and output f - R is complete.
//
// NONORTH adds the mixed terms of the Laplacian (Hamiltonian.cpp:176-267),
//   sum_pq cxy[p] d1y[q] (x(+p,+q) - x(+p,-q) - x(-p,+q) + x(-p,-q))  (x,y)
// and the same for (x,z) and (y,z), each factored into two antisymmetric
// sums: xy: sum_p cxy[p] (g(x+p) - g(x-p)) with g = sum_q d1y[q] (x(y+q) -
// x(y-q)), which returns to LDS (with x ghosts) and is read one plane later;
// xz + yz: sum_q d1z[q] (h(z+q) - h(z-q)) with h = sum_p cxz[p] (x(x+p) -
// x(x-p)) + cyz[p] (x(y+p) - x(y-p)), which joins the forward accumulation:
// 36 LDS reads and about 60 FMAs instead of 108 four-point groups.
//
// LDS: two plane buffers of band rows plus R rows above and below, R ghost
// columns on each side (wrapped copies times the Bloch factor of the face,
// HaloExchange.cpp:104-189), the row pitch W a compile-time constant so that
// a neighbour is one address plus an immediate offset; NONORTH two planes of
// g.  Halo rows carry no ghost columns (the mixed terms go through g).  One
// barrier per plane.
//
// WRAPZ: the workgroup owns the whole periodic z range and marches its nz
// planes once instead of nz + 2R wrapped ones: the R outputs at each end then
// lack the planes across the z boundary.  The first 2R steps put the wrapped
// part of the bottom outputs and the top outputs without theirs into LDS (2R
// values per thread); after the march the accumulators hold the other parts.
//
// What bounds it: instruction issue, then LDS and barrier latency (112 units
// of 24^3 x 12 complex64: about 110 of 172 us are vector instructions).  Hence
// one point per thread (runs of two double the registers: 244 us), and no
// branch or scalar load in the loop that can be outside it: lanes and halo
// slots beyond the band repeat its last point, the Bloch factors of a lane's
// ghost and halo copies are picked once, and WRAPZ has no test for a plane
// beyond the boundary.  With these as branches and loads in the loop, and the
// end planes' partial sums in memory, the same step took 297 us; complex128
// 553 us, now 305 us (892 MB: 2.9 TB/s).  Alone: 48^3 x 64 double skew 93 ->
// 69 us, 40^3 x 48 complex128 orthogonal 75 -> 47 us.
// Real orthogonal blocks that the run-vector kernel does not take, and all of
// them in batches: 25 x 27 x 29 x 1600 double 311 -> 209 us against several
// points per thread; batches of 24..40^3 frames, 15.3 M points in all, step of
// double 600 us as 16-byte runs, now 568 us (all launches of a step).
template <class S, bool NONORTH, bool WRAPZ, int HP, int W>
__device__ __forceinline__ void stencil_points_body(const NonorthArgs<typename Tr<S>::A> &q,
                                                    const StepIO<typename Tr<S>::A> io, const int w)
{
    using A = typename Tr<S>::A;
    constexpr bool C = Tr<S>::C;
    constexpr int R = kMaxR, NA = 2 * R + 1;
    const StepArgs<A> &p = q.b;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int NT = blockDim.x, tid = threadIdx.x;
    const int xplane = W * (p.tyr + 2 * R), gplane = W * p.tyr;
    S *const ldsx = reinterpret_cast<S *>(smem_raw);
    S *const ldsg = ldsx + 2 * xplane;
    S *const stash = ldsg + (NONORTH ? 2 * gplane : 0) + tid;

    const int band = w % p.nbands;
    const int rest = w / p.nbands;
    const int zc = rest % p.nzch;
    const int col = rest / p.nzch;
    const int y0 = band * p.tyr;
    const int rows = min(p.tyr, ny - y0);
    const int z0 = zc * p.zch;
    const int z1 = min(z0 + p.zch, nz);
    const int nxny = nx * ny;
    const S *__restrict__ X = global_ptr(reinterpret_cast<const S *>(io.x)) + (long)col * io.ldx;
    const S *__restrict__ O = global_ptr(reinterpret_cast<const S *>(io.old)) + (long)col * io.ldo;
    S *__restrict__ Y = global_ptr(reinterpret_cast<S *>(io.out)) + (long)col * io.ldout;
    const A *__restrict__ Vf = global_ptr(p.veff);
    const bool has_old = io.old != nullptr && io.b != A(0);   // no Y_(k-2) stream without a buffer

    // the owned point; lanes beyond the band repeat its last one (and write
    // the same values to LDS), all but the store of the result
    const bool own = tid < rows * nx;
    const int qt = own ? tid : rows * nx - 1;
    const int yy = qt / nx;
    const int x0 = qt - yy * nx;
    const unsigned off = (y0 + yy) * nx + x0;
    const int li = (yy + R) * W + R + x0;
    const int gi = yy * W + R + x0;
    // its copy in the ghost columns: at x + nx from the left face, x - nx from
    // the right one, with the Bloch factor of the face crossed (rows shorter
    // than 2R: both)
    const bool gx = x0 < R || x0 >= nx - R;
    const int gxs = x0 < R ? nx : -nx;
    const bool gx2 = x0 < R && x0 >= nx - R;
    A gxr = A(1), gxi = A(0);
    if constexpr (C) {
        gxr = p.ph[0][x0 < R][0];
        gxi = p.ph[0][x0 < R][1];
    }
    // halo points: R rows below and R above the band, wrapped in y; slots
    // beyond the last repeat it
    unsigned hoff[HP];
    int hli[HP];
    A hr[HP], hi[HP];
#pragma unroll
    for (int h = 0; h < HP; ++h) {
        const int t = min(tid + h * NT, 2 * R * nx - 1);
        const int i = t / nx;
        const int xx = t - i * nx;
        const int yb = i < R ? i - R : rows + i - R;
        int yg = y0 + yb;
        hr[h] = A(1);
        hi[h] = A(0);
        if constexpr (C) {
            if (yg < 0 || yg >= ny) {
                hr[h] = p.ph[1][yg >= ny][0];
                hi[h] = p.ph[1][yg >= ny][1];
            }
        }
        if (yg < 0) yg += ny;
        else if (yg >= ny) yg -= ny;
        hoff[h] = yg * nx + xx;
        hli[h] = (yb + R) * W + R + xx;
    }

    const int f_end = WRAPZ ? z1 - 1 : z1 - 1 + R;
    // planes beyond the chunk feed z-terms only, unless their h is needed
    auto inplane = [&](int f) { return NONORTH || WRAPZ || (f >= z0 && f < z1); };
    // every load of plane f (owned and halo points, z-wrapped, and Veff) and
    // of the output plane f - R (Y_{k-2}), clamped into range
    auto issue = [&](int f, PointLoads<S, HP> &L) {
        f = min(f, f_end);
        int zz = f;
        if (zz < 0) zz += nz;
        else if (zz >= nz) zz -= nz;
        const S *Xz = X + zz * nxny;
        L.front = ld_at(Xz, off);
        if (inplane(f)) {
#pragma unroll
            for (int h = 0; h < HP; ++h) L.halo[h] = ld_at(Xz, hoff[h]);
        }
        if (has_old) L.old = ld_at(O + max(f - R, WRAPZ ? R : z0) * nxny, off);
        L.v = ld_at(Vf + min(max(f, z0), z1 - 1) * nxny, off);
    };

    // acc[j]: -2 (H - s) x at output plane f - R + j, so H x = -acc / 2
    S acc[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) acc[j] = zero<S>();
    const A diag = NONORTH ? (q.beta[0] + q.beta[1] + q.beta[2]) * q.w2[0] : p.c[0][0] + p.c[1][0] + p.c[2][0];

    auto put = [&](S *L, int i, S v) {   // a value and its ghost columns
        L[i] = v;
        if (gx) L[i + gxs] = phased(v, gxr, gxi);
        if (nx < 2 * R && gx2) L[i - nx] = phased(v, p.ph[0][0][0], p.ph[0][0][1]);
    };
    // xy term from a complete g plane
    auto mixed_xy = [&](const S *LG, S a) {
        S m = zero<S>();
#pragma unroll
        for (int k = 1; k <= R; ++k) m = fm(q.w1[k], add(LG[gi + k], scl(A(-1), LG[gi - k])), m);
        return fm(q.axy_hy, m, a);
    };

    int buf = 0;
    auto step = [&](int f, PointLoads<S, HP> &cur, PointLoads<S, HP> &nxt) {
        __builtin_amdgcn_sched_barrier(0);
        issue(f + 1, nxt);
        S xf = cur.front, hz = zero<S>();
        // Bloch factor of a plane beyond the z boundary (uniform)
        A zr = A(1), zi = A(0);
        const bool zph = C && !WRAPZ && (f < 0 || f >= nz);
        if (zph) {
            zr = p.ph[2][f >= nz][0];
            zi = p.ph[2][f >= nz][1];
            xf = phased(xf, zr, zi);
        }
        if (inplane(f)) {
            S *LX = ldsx + buf * xplane;
            put(LX, li, xf);
#pragma unroll
            for (int h = 0; h < HP; ++h) {
                S t = phased(cur.halo[h], hr[h], hi[h]);
                if (zph) t = phased(t, zr, zi);
                LX[hli[h]] = t;
            }
            __syncthreads();
            if constexpr (NONORTH) {
                if (WRAPZ ? f > z0 : f - 1 >= z0 && f - 1 < z1)
                    acc[R - 1] = mixed_xy(ldsg + (buf ^ 1) * gplane, acc[R - 1]);
                // x, then y neighbours; the scheduling barriers keep the
                // compiler from hoisting all LDS reads at once (registers)
                __builtin_amdgcn_sched_barrier(0);
                S sx2 = zero<S>(), sx1 = zero<S>(), sy2 = zero<S>(), sy1 = zero<S>();
#pragma unroll
                for (int k = 1; k <= R; ++k) {
                    const S xp = LX[li + k], xm = LX[li - k];
                    sx2 = fm(q.w2[k], add(xp, xm), sx2);
                    sx1 = fm(q.w1[k], add(xp, scl(A(-1), xm)), sx1);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 1; k <= R; ++k) {
                    const S yp = LX[li + k * W], ym = LX[li - k * W];
                    sy2 = fm(q.w2[k], add(yp, ym), sy2);
                    sy1 = fm(q.w1[k], add(yp, scl(A(-1), ym)), sy1);
                }
                put(ldsg + buf * gplane, gi, sy1);
                const S a2 = fm(diag - A(2) * (cur.v + io.s), xf, scl(q.beta[0], sx2));
                acc[R] = add(acc[R], fm(q.beta[1], sy2, a2));
                hz = scl(q.ihz, fm(q.axz, sx1, scl(q.ayz, sy1)));
            } else {
                S s = fm(diag - A(2) * (cur.v + io.s), xf, acc[R]);
#pragma unroll
                for (int k = 1; k <= R; ++k) {
                    s = fm(p.c[0][k], add(LX[li + k], LX[li - k]), s);
                    s = fm(p.c[1][k], add(LX[li + k * W], LX[li - k * W]), s);
                    if (C && k % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                }
                acc[R] = s;
            }
            buf ^= 1;
        }
        // z-terms of plane f for outputs f - R + j, j != R
        const S xz = NONORTH ? scl(q.beta[2], xf) : xf;
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            if (j == R) continue;
            const int d = j < R ? R - j : j - R;
            if constexpr (NONORTH) {
                acc[j] = fm(q.w2[d], xz, acc[j]);
                acc[j] = fm(j < R ? q.w1[d] : -q.w1[d], hz, acc[j]);
            } else {
                acc[j] = fm(p.c[2][d], xz, acc[j]);
            }
        }
        const int fo = f - R;
        if (WRAPZ && fo < R) {
            stash[f * NT] = acc[0];
        } else if (fo >= z0) {
            S res = scl(A(-0.5) * io.a, acc[0]);
            if (has_old) res = fm(io.b, cur.old, res);
            if (own) st_at(Y + fo * nxny, off, res);
        }
#pragma unroll
        for (int j = 0; j + 1 < NA; ++j) acc[j] = acc[j + 1];
        acc[NA - 1] = zero<S>();
    };

    // two load sets in turn; the test between the two steps keeps the compiler
    // from merging them (20 to 40 registers more, spills in complex128)
    PointLoads<S, HP> la, lb;
    int f = WRAPZ ? z0 : z0 - R;
    issue(f, la);
    for (; f <= f_end; f += 2) {
        step(f, la, lb);
        if (f + 1 <= f_end) step(f + 1, lb, la);
    }
    if constexpr (!WRAPZ) return;
    if constexpr (NONORTH) {
        // the xy term of the last plane
        __syncthreads();
        acc[R - 1] = mixed_xy(ldsg + (buf ^ 1) * gplane, acc[R - 1]);
    }
    if (!own) return;
    // the 2R end outputs: acc[j] and stash j hold the two parts of output
    // nz - R + j (j < R) or j - R, the part across the boundary with its
    // Bloch factor; a group's loads are all in flight before its first store
    constexpr int G = sizeof(S) <= 8 ? 2 * R : R;
#pragma unroll
    for (int j0 = 0; j0 < 2 * R; j0 += G) {
        S t[G];
        if (has_old) {
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int j = j0 + i;
                t[i] = ld_at(O + (j < R ? nz - R + j : j - R) * nxny, off);
            }
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const int j = j0 + i;
            S c = stash[j * NT], d = acc[j];
            if (j < R) c = phased(c, p.ph[2][1][0], p.ph[2][1][1]);
            else d = phased(d, p.ph[2][0][0], p.ph[2][0][1]);
            S res = scl(A(-0.5) * io.a, add(c, d));
            if (has_old) res = fm(io.b, t[i], res);
            st_at(Y + (j < R ? nz - R + j : j - R) * nxny, off, res);
        }
    }
}

template <class S, bool NONORTH, bool WRAPZ, int HP, int W>
__global__ void __launch_bounds__(512) k_stencil_points(NonorthArgs<typename Tr<S>::A> q)
{
    const int w = xcd_work_item();
    if (w >= q.b.nwork) return;
    stencil_points_body<S, NONORTH, WRAPZ, HP, W>(q, step_io(q.b), w);
}

template <class S, bool NONORTH, bool WRAPZ, int HP, int W>
__global__ void __launch_bounds__(512) k_stencil_points_batch(const BatchRec<typename Tr<S>::A> *__restrict__ recs,
                                                              const int *__restrict__ item_unit, int nitems,
                                                              const typename Tr<S>::A *__restrict__ coef, int ix,
                                                              int iold, int iout)
{
    using A = typename Tr<S>::A;
    const int w = xcd_work_item();
    if (w >= nitems) return;
    const int u = item_unit[w];
    const BatchRec<A> &r = recs[u];
    const StepIO<A> io{r.buf[ix], r.buf[iold], const_cast<void *>(r.buf[iout]), r.ld[ix], r.ld[iold], r.ld[iout],
                       coef[3 * u], coef[3 * u + 1], coef[3 * u + 2]};
    const NonorthArgs<A> q = r.q;
    stencil_points_body<S, NONORTH, WRAPZ, HP, W>(q, io, w - r.item0);
}

// The kernels of a shape: f(nonorth, wrapz, halo slots, pitch) as constants.
template <class F>
void by_point_shape(const PointShape &s, bool nonorth, F &&f)
{
    auto pitch = [&](auto no, auto wz) {
        auto halo = [&](auto w, auto lo, auto mid, auto hi) {
            if (s.hp <= decltype(lo)::value) f(no, wz, lo, w);
            else if (s.hp <= decltype(mid)::value) f(no, wz, mid, w);
            else f(no, wz, hi, w);
        };
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        using I6 = std::integral_constant<int, 6>;
        switch (s.pitch) {
            case 40: halo(std::integral_constant<int, 40>{}, I1{}, I2{}, I2{}); break;
            case 64: halo(std::integral_constant<int, 64>{}, I2{}, I3{}, I3{}); break;
            case 76: halo(std::integral_constant<int, 76>{}, I2{}, I3{}, I3{}); break;
            case 128: halo(std::integral_constant<int, 128>{}, I2{}, I3{}, I6{}); break;
            default: f(no, wz, I6{}, std::integral_constant<int, 256>{}); break;
        }
    };
    auto wrap = [&](auto no) {
        if (s.wrapz) pitch(no, std::true_type{});
        else pitch(no, std::false_type{});
    };
    if (nonorth) wrap(std::true_type{});
    else wrap(std::false_type{});
}

template <class S>
void launch_points(const StencilGeom &g, const void *x, long ldx, const void *old, long ldo, void *out, long ldout,
                   const void *veff, int ncol, double a, double b, double s, const PointShape &sh, hipStream_t st,
                   const void *coef)
{
    using A = typename Tr<S>::A;
    NonorthArgs<A> q = operator_args<A>(g);
    StepArgs<A> &p = q.b;
    p.x = x; p.old = old; p.out = out; p.veff = static_cast<const A *>(veff);
    p.ldx = ldx; p.ldo = ldo; p.ldout = ldout;
    p.ncol = ncol;
    p.lpr = 0;
    p.tyr = sh.tyr;
    p.nbands = (g.ny + sh.tyr - 1) / sh.tyr;
    p.zch = (g.nz + sh.nzch - 1) / sh.nzch;
    p.nzch = (g.nz + p.zch - 1) / p.zch;
    p.nwork = p.nbands * p.nzch * ncol;
    p.a = (A)a; p.b = (A)b; p.s = (A)s;
    p.coef = static_cast<const A *>(coef);
    const int blocks = ((p.nwork + 7) / 8) * 8;
    by_point_shape(sh, !g.orth, [&](auto no, auto wz, auto hp, auto w) {
        hipLaunchKernelGGL((k_stencil_points<S, decltype(no)::value, decltype(wz)::value, decltype(hp)::value,
                                             decltype(w)::value>),
                           dim3(blocks), dim3(sh.nt), sh.lds, st, q);
    });
}

template <class S>
void launch_points_batch(const void *recs, const int *items, int nitems, bool nonorth, const void *coef, int ix,
                         int iold, int iout, const PointShape &sh, hipStream_t st)
{
    using A = typename Tr<S>::A;
    const int blocks = ((nitems + 7) / 8) * 8;
    by_point_shape(sh, nonorth, [&](auto no, auto wz, auto hp, auto w) {
        hipLaunchKernelGGL((k_stencil_points_batch<S, decltype(no)::value, decltype(wz)::value, decltype(hp)::value,
                                                   decltype(w)::value>),
                           dim3(blocks), dim3(sh.nt), sh.lds, st, static_cast<const BatchRec<A> *>(recs), items,
                           nitems, static_cast<const A *>(coef), ix, iold, iout);
    });
}

}  // namespace
}  // namespace gpu
}  // namespace lynx

// Defines the launches of element type S under the names points_step_<tag>
// and points_batch_<tag>.
#define LYNX_POINTS(S, tag)                                                                                     \
    namespace lynx {                                                                                            \
    namespace gpu {                                                                                             \
    void points_step_##tag(const StencilGeom &g, const void *x, long ldx, const void *old, long ldo, void *out, \
                           long ldout, const void *veff, int ncol, double a, double b, double s,                \
                           const PointShape &sh, hipStream_t st, const void *coef)                              \
    {                                                                                                           \
        launch_points<S>(g, x, ldx, old, ldo, out, ldout, veff, ncol, a, b, s, sh, st, coef);                   \
    }                                                                                                           \
    void points_batch_##tag(const void *recs, const int *items, int nitems, bool nonorth, const void *coef,     \
                            int ix, int iold, int iout, const PointShape &sh, hipStream_t st)                   \
    {                                                                                                           \
        launch_points_batch<S>(recs, items, nitems, nonorth, coef, ix, iold, iout, sh, st);                     \
    }                                                                                                           \
    }                                                                                                           \
    }
