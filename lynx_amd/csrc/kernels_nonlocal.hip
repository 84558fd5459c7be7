// Nonlocal projector gather, alone or behind the scatter of the step before,
// on the matrix cores.
#include "kernels_nonlocal.hpp"
#include "stencil_common.hpp"

#include <algorithm>
#include <string>

namespace lynx {
namespace gpu {
namespace {

// 16 x 16 products of K = 4 in the arithmetic type, the result row of
// element v in lane group l / 16 (its column is l % 16), and the complex
// column of a row when rows are the real and imaginary parts of 8 complex
// columns, chosen so that a lane holds both parts (elements 2h and 2h + 1).
template <class A> struct Mma;
template <> struct Mma<double> {
    typedef double V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V mma(double a, double b, V c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int group, int v) { return group + 4 * v; }
    static __device__ __forceinline__ int ccol(int row) { return (row & 3) + 4 * (row >> 3); }
    static __device__ __forceinline__ int cpart(int row) { return (row >> 2) & 1; }
};
template <> struct Mma<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V mma(float a, float b, V c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int group, int v) { return 4 * group + v; }
    static __device__ __forceinline__ int ccol(int row) { return row >> 1; }
    static __device__ __forceinline__ int cpart(int row) { return row & 1; }
};

// elements of a wave's LDS slab: a 16 x 16 tile of pitch 17, later its sums
template <int NPM> constexpr int slab_elems() { return NPM > 16 ? 512 : 272; }

// One workgroup per (atom, group of 16 real or 8 complex columns).  A wave
// takes tiles of 16 sphere points: lane l holds point l % 16 of the columns
// row(l / 16, v), so an access covers 16 consecutive points (chords of the
// sphere) of four columns.  The scatter's product (columns x points, K =
// projectors) arrives in that layout; y is updated and stored; the tile is
// transposed through the wave's LDS slab, and the gather's product
// (projectors x columns, K = points) takes it four points at a time.  The
// waves' sums are added in wave order through LDS.
//
// Bound by the partial cache lines of y (a chord is 32 to 128 bytes), then by
// the latency of a tile's two dependent loads (index, value); hence one pass
// for the scatter of a step and the gather of the next, about two tiles to a
// wave, and as many waves as that needs.  Against a gather with a wave per
// (atom, column), whose lane exchanges took as long as its loads, and a
// scatter apart: 64 atoms x 160 columns of 60^3 double 39 us (60 us); 216
// atoms x 480 of 90^3 float 250 us (323 us); 14 atoms x 48 of 40^3
// complex128 8 us (17 us); 8 atoms x 24 of 30^3 double 8 us (11 us and a
// launch).  With lanes holding columns instead of points (no transposition)
// the stores broke the chords up: 45 us, 404 us, 9 us, 10 us.
template <class S, int NPM, int MODE, class T>
__device__ __forceinline__ void nl_tile_body(const NlArgs<typename Tr<S>::A> &p, const S *__restrict__ beta_in,
                                             S *__restrict__ beta_out, T *Y, long ldy, int ncol, typename Tr<S>::A a,
                                             int at, int cg)
{
    using A = typename Tr<S>::A;
    using M = Mma<A>;
    using V = typename M::V;
    constexpr bool C = Tr<S>::C, SCATTER = MODE == kNlUpdate;
    constexpr int MT = (NPM + 15) / 16, KS = NPM / 4, CW = C ? 2 : 1, NV = 4 / CW;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int lc = lane & 15, lg = lane >> 4;
    A *const slab = reinterpret_cast<A *>(smem_raw) + wave * slab_elems<NPM>();
    const int c0 = cg * (16 / CW);
    // the lane's columns of y: elements v (real) or pairs (complex)
    T *y[NV];
    bool cv[NV];
#pragma unroll
    for (int h = 0; h < NV; ++h) {
        const int col = c0 + (C ? M::ccol(M::row(lg, 2 * h)) : M::row(lg, h));
        cv[h] = col < ncol;
        y[h] = Y + (long)min(col, ncol - 1) * ldy;
    }
    // as matrix row or column, lane index lc stands for this column
    const int mc = min(c0 + (C ? M::ccol(lc) : lc), ncol - 1), mp = C ? M::cpart(lc) : 0;
    const int pb = p.atom_pt_off[at], pe = p.atom_pt_off[at + 1];
    A b[KS];
    if constexpr (SCATTER) {
#pragma unroll
        for (int k = 0; k < KS; ++k)
            b[k] = reinterpret_cast<const A *>(beta_in)[(((long)mc * p.n_atom + at) * NPM + lg + 4 * k) * CW + mp];
    }
    V acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = V{A(0), A(0), A(0), A(0)};
    for (int p0 = pb + 16 * wave; p0 < pe; p0 += 16 * nw) {
        const bool in = p0 + lc < pe;
        const int q = in ? p0 + lc : pe - 1;
        const long g = p.pt_gpos[q];
        A pr = A(1), pi = A(0);
        if constexpr (C) {
            const int im = p.pt_img[q];
            pr = p.phase[2 * im];
            pi = p.phase[2 * im + 1];
        }
        S x[NV];
#pragma unroll
        for (int h = 0; h < NV; ++h) x[h] = to_compute(y[h][g]);
        V s = V{A(0), A(0), A(0), A(0)};
        if constexpr (SCATTER) {
#pragma unroll
            for (int k = 0; k < KS; ++k) s = M::mma(b[k], p.chi[(long)q * NPM + lg + 4 * k], s);
        }
        A ch[MT][4];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int pt = p0 + lg + 4 * v, j = 16 * m + lc;
                const A t = p.chi[(long)min(pt, pe - 1) * NPM + min(j, NPM - 1)];
                ch[m][v] = pt < pe && j < NPM ? t : A(0);
            }
#pragma unroll
        for (int h = 0; h < NV; ++h) {
            if constexpr (SCATTER) {
                S t;
                if constexpr (C) t = cmul(S{s[2 * h], s[2 * h + 1]}, pr, -pi);
                else t = s[h];
                const T r = StoreAs<T>::from(fm(a, t, x[h]));
                if (in && cv[h]) y[h][g] = r;
                x[h] = to_compute(r);
            }
            x[h] = phased(x[h], pr, pi);
            // a lane beyond the sphere repeats its last point: its value
            // must not reach the product (0 times infinity)
            if (!in) x[h] = zero<S>();
            if constexpr (C) {
                slab[lc * 17 + M::row(lg, 2 * h)] = x[h].x;
                slab[lc * 17 + M::row(lg, 2 * h + 1)] = x[h].y;
            } else {
                slab[lc * 17 + M::row(lg, h)] = x[h];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const A t = slab[(lg + 4 * v) * 17 + lc];
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = M::mma(ch[m][v], t, acc[m]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) slab[m * 256 + lane * 4 + v] = acc[m][v];
    __syncthreads();
    for (int i = threadIdx.x; i < MT * 256; i += blockDim.x) {
        const int v = i & 3, ln = (i >> 2) & 63, m = i >> 8;
        const int j = 16 * m + M::row(ln >> 4, v), n = ln & 15;
        const int c = c0 + (C ? M::ccol(n) : n);
        if (j >= NPM || c >= ncol) continue;
        const A *r = reinterpret_cast<const A *>(smem_raw) + i;
        A t = A(0);
        for (int w = 0; w < nw; ++w) t += r[w * slab_elems<NPM>()];
        reinterpret_cast<A *>(beta_out)[(((long)c * p.n_atom + at) * NPM + j) * CW + (C ? M::cpart(n) : 0)] =
            p.gamma[at * NPM + j] * t;
    }
}

template <class S, int NPM, int MODE, class T>
__global__ void __launch_bounds__(1024) k_nl_tile(NlArgs<typename Tr<S>::A> p, const S *__restrict__ beta_in,
                                                  S *__restrict__ beta_out, T *Y, long ldy, int ncol,
                                                  typename Tr<S>::A a, const typename Tr<S>::A *acoef)
{
    if (acoef) a = acoef[0];
    nl_tile_body<S, NPM, MODE, T>(p, beta_in, beta_out, Y, ldy, ncol, a, blockIdx.x, blockIdx.y);
}

template <class S, int NPM, int MODE>
__global__ void __launch_bounds__(1024) k_nl_tile_batch(const BatchRec<typename Tr<S>::A> *__restrict__ recs,
                                                        const int *__restrict__ item_unit, int nitems,
                                                        const S *__restrict__ beta_in, S *__restrict__ beta_out,
                                                        const typename Tr<S>::A *__restrict__ coef, int iy)
{
    const int w = blockIdx.x;
    if (w >= nitems) return;
    const int u = item_unit[w];
    const BatchRec<typename Tr<S>::A> &r = recs[u];
    const int lb = w - r.g_item0;
    nl_tile_body<S, NPM, MODE, S>(global_args(r.nl), beta_in + r.beta_off, beta_out + r.beta_off,
                                  global_ptr(reinterpret_cast<S *>(const_cast<void *>(r.buf[iy]))), r.ld[iy], r.ncol,
                                  coef[3 * u], lb % r.nl.n_atom, lb / r.nl.n_atom);
}

template <class F>
void by_npm(int npm, F &&f)
{
    if (npm == 8) f(std::integral_constant<int, 8>{});
    else if (npm == 16) f(std::integral_constant<int, 16>{});
    else f(std::integral_constant<int, 32>{});
}
template <class F>
void by_mode(NlMode mode, F &&f)
{
    if (mode == kNlGather) f(std::integral_constant<int, kNlGather>{});
    else f(std::integral_constant<int, kNlUpdate>{});
}

// LDS of the waves' slabs
size_t tile_lds(int e, int npm, int waves)
{
    const size_t n = npm > 16 ? slab_elems<32>() : slab_elems<16>();
    return waves * n * (elem_single(e) ? 4 : 8);
}

}  // namespace

bool nl_tile_fits(const NlDev &nl, NlMode mode)
{
    return nl.max_atom_pts <= kTileAtomPts && (mode == kNlGather || nl.disjoint);
}

int nl_tile_groups(int e, int ncol)
{
    const int per = elem_complex(e) ? 8 : 16;
    return (ncol + per - 1) / per;
}

int nl_tile_waves(int max_atom_pts) { return std::max(1, std::min(16, (max_atom_pts + 31) / 32)); }

void nl_tile(int e, const NlDev &nl, NlMode mode, const void *beta_in, void *beta_out, void *y, long ldy, int ncol,
             double a, hipStream_t st, const void *acoef)
{
    if (nl.n_atom == 0 || nl.n_pts == 0) return;
    const int waves = nl_tile_waves(nl.max_atom_pts);
    const dim3 grid(nl.n_atom, nl_tile_groups(e, ncol));
    const size_t lds = tile_lds(e, nl.npm, waves);
    by_npm(nl.npm, [&](auto np) {
        by_mode(mode, [&](auto md) {
            auto go = [&](auto s, auto t) {
                using S = decltype(s);
                using T = decltype(t);
                using A = typename Tr<S>::A;
                const NlArgs<A> p{nl.atom_pt_off, nl.pt_gpos, nl.pt_img, nl.pt_atom, nl.cov_off, nl.cov_gpos,
                                  nl.ent_pt, (const A *)nl.chi, (const A *)nl.gamma, (const A *)nl.phase, nl.n_atom,
                                  nl.n_cov, nl.npm};
                hipLaunchKernelGGL((k_nl_tile<S, decltype(np)::value, decltype(md)::value, T>), grid, dim3(64 * waves),
                                   lds, st, p, (const S *)beta_in, (S *)beta_out, (T *)y, ldy, ncol, (A)a,
                                   (const A *)acoef);
            };
            switch (e) {
                case F64: go(double{}, double{}); break;
                case C128: go(double2{}, double2{}); break;
                case F32: go(float{}, float{}); break;
                case C64: go(float2{}, float2{}); break;
                default: go(float{}, bf16{}); break;
            }
        });
    });
}

void nl_tile_batch(int e, int npm, const void *recs, const int *items, int nitems, int waves, NlMode mode,
                   const void *beta_in, void *beta_out, const void *coef, int iy, hipStream_t st)
{
    const size_t lds = tile_lds(e, npm, waves);
    by_npm(npm, [&](auto np) {
        by_mode(mode, [&](auto md) {
            auto go = [&](auto s) {
                using S = decltype(s);
                using A = typename Tr<S>::A;
                hipLaunchKernelGGL((k_nl_tile_batch<S, decltype(np)::value, decltype(md)::value>), dim3(nitems),
                                   dim3(64 * waves), lds, st, static_cast<const BatchRec<A> *>(recs), items, nitems,
                                   (const S *)beta_in, (S *)beta_out, static_cast<const A *>(coef), iy);
            };
            switch (e) {
                case F64: go(double{}); break;
                case C128: go(double2{}); break;
                case F32: go(float{}); break;
                default: go(float2{}); break;
            }
        });
    });
}

}  // namespace gpu
}  // namespace lynx
