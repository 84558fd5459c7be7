// Device-side pieces shared by the stencil and nonlocal kernels: element
// types, operator records and addressing helpers.  Included by HIP sources
// only.
#pragma once

#include "kernels.hpp"
#include "common.hpp"

#include <hip/hip_runtime.h>
#include <cstdint>
#include <type_traits>

namespace lynx {
namespace gpu {
namespace {

// ------------------------------------------------------------ element ops --
template <class S> struct Tr;
template <> struct Tr<double> { using A = double; static constexpr bool C = false; };
template <> struct Tr<float> { using A = float; static constexpr bool C = false; };
template <> struct Tr<double2> { using A = double; static constexpr bool C = true; };
template <> struct Tr<float2> { using A = float; static constexpr bool C = true; };

// the FP64 type of each element type (partial sums of single-precision
// products are added in double precision)
template <class S> struct Wide { using T = S; };
template <> struct Wide<float> { using T = double; };
template <> struct Wide<float2> { using T = double2; };
__device__ __forceinline__ double widen(double x) { return x; }
__device__ __forceinline__ double widen(float x) { return (double)x; }
__device__ __forceinline__ double2 widen(double2 x) { return x; }
__device__ __forceinline__ double2 widen(float2 x) { return make_double2(x.x, x.y); }

// bfloat16 storage (the filter's BF16 mode): 8-bit mantissa in memory,
// arithmetic in float.  Conversion to float is exact; from float it rounds
// to nearest even (finite values).
struct bf16 {
    unsigned short b;
};
__device__ __forceinline__ float to_compute(bf16 v) { return __uint_as_float((unsigned)v.b << 16); }
__device__ __forceinline__ float to_compute(float v) { return v; }
__device__ __forceinline__ double to_compute(double v) { return v; }
__device__ __forceinline__ double2 to_compute(double2 v) { return v; }
__device__ __forceinline__ float2 to_compute(float2 v) { return v; }
template <class T> struct StoreAs;
template <> struct StoreAs<bf16> {
    static __device__ __forceinline__ bf16 from(float f)
    {
        return __builtin_bit_cast(bf16, (__bf16)f);   // v_cvt_pk_bf16_f32
    }
};
template <> struct StoreAs<float> { static __device__ __forceinline__ float from(float f) { return f; } };
template <> struct StoreAs<double> { static __device__ __forceinline__ double from(double f) { return f; } };
template <> struct StoreAs<float2> { static __device__ __forceinline__ float2 from(float2 f) { return f; } };
template <> struct StoreAs<double2> { static __device__ __forceinline__ double2 from(double2 f) { return f; } };

template <class S> __device__ __forceinline__ S zero();
template <> __device__ __forceinline__ double zero<double>() { return 0.0; }
template <> __device__ __forceinline__ float zero<float>() { return 0.0f; }
template <> __device__ __forceinline__ double2 zero<double2>() { return make_double2(0.0, 0.0); }
template <> __device__ __forceinline__ float2 zero<float2>() { return make_float2(0.0f, 0.0f); }

__device__ __forceinline__ double add(double a, double b) { return a + b; }
__device__ __forceinline__ float add(float a, float b) { return a + b; }
__device__ __forceinline__ double2 add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }

// scalar * element
__device__ __forceinline__ double scl(double a, double x) { return a * x; }
__device__ __forceinline__ float scl(float a, float x) { return a * x; }
__device__ __forceinline__ double2 scl(double a, double2 x) { return make_double2(a * x.x, a * x.y); }
__device__ __forceinline__ float2 scl(float a, float2 x) { return make_float2(a * x.x, a * x.y); }

// a * x + y with scalar a
__device__ __forceinline__ double fm(double a, double x, double y) { return fma(a, x, y); }
__device__ __forceinline__ float fm(float a, float x, float y) { return fmaf(a, x, y); }
__device__ __forceinline__ double2 fm(double a, double2 x, double2 y) { return make_double2(fma(a, x.x, y.x), fma(a, x.y, y.y)); }
__device__ __forceinline__ float2 fm(float a, float2 x, float2 y) { return make_float2(fmaf(a, x.x, y.x), fmaf(a, x.y, y.y)); }

// x * (pr + i pi)
__device__ __forceinline__ double2 cmul(double2 x, double pr, double pi)
{
    return make_double2(x.x * pr - x.y * pi, x.x * pi + x.y * pr);
}
__device__ __forceinline__ float2 cmul(float2 x, float pr, float pi)
{
    return make_float2(x.x * pr - x.y * pi, x.x * pi + x.y * pr);
}
template <class S, class A>
__device__ __forceinline__ S phased(S v, A pr, A pi)
{
    if constexpr (Tr<S>::C) return cmul(v, pr, pi);
    else return v;
}

// conj(a) * b and its accumulation
__device__ __forceinline__ double cfma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float cfma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c)
{
    return make_double2(fma(a.x, b.x, fma(a.y, b.y, c.x)), fma(a.x, b.y, fma(-a.y, b.x, c.y)));
}
__device__ __forceinline__ float2 cfma(float2 a, float2 b, float2 c)
{
    return make_float2(fmaf(a.x, b.x, fmaf(a.y, b.y, c.x)), fmaf(a.x, b.y, fmaf(-a.y, b.x, c.y)));
}
// a * b + c (complex)
__device__ __forceinline__ double mfma_(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float mfma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double2 mfma_(double2 a, double2 b, double2 c)
{
    return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ float2 mfma_(float2 a, float2 b, float2 c)
{
    return make_float2(fmaf(a.x, b.x, fmaf(-a.y, b.y, c.x)), fmaf(a.x, b.y, fmaf(a.y, b.x, c.y)));
}

__device__ __forceinline__ double re2(double a) { return a * a; }
__device__ __forceinline__ double re2(float a) { return double(a) * a; }
__device__ __forceinline__ double re2(double2 a) { return a.x * a.x + a.y * a.y; }
__device__ __forceinline__ double re2(float2 a) { return double(a.x) * a.x + double(a.y) * a.y; }
__device__ __forceinline__ double redot(double a, double b) { return a * b; }
__device__ __forceinline__ double redot(float a, float b) { return double(a) * b; }
__device__ __forceinline__ double redot(double2 a, double2 b) { return a.x * b.x + a.y * b.y; }
__device__ __forceinline__ double redot(float2 a, float2 b) { return double(a.x) * b.x + double(a.y) * b.y; }

// -------------------------------------------------------- operator records --
template <class A>
struct StepArgs {
    const void *x;
    const void *old;
    void *out;
    const A *veff;
    long ldx, ldo, ldout;
    int nx, ny, nz, ncol;
    int tyr, nbands, zch, nzch, nwork;
    int lpr;            // 16-byte-run kernels: lanes per band row (>= runs per row)
    A c[3][kMaxR + 1];
    A a, b, s;
    A ph[3][2][2];
    // when set, (a, b, s) are read from this device triple instead (the
    // filter's steps in a replayed HIP graph take their scalars from a
    // table uploaded per call)
    const A *coef = nullptr;
};

// Per-launch operands of a step (buffers and recurrence scalars), kept
// apart from the operator record so that a batch can read the record from
// device memory while these arrive as kernel arguments.
template <class A>
struct StepIO {
    const void *x;
    const void *old;
    void *out;
    long ldx, ldo, ldout;
    A a, b, s;
};

template <class A>
__device__ inline StepIO<A> step_io(const StepArgs<A> &p)
{
    if (p.coef) return StepIO<A>{p.x, p.old, p.out, p.ldx, p.ldo, p.ldout, p.coef[0], p.coef[1], p.coef[2]};
    return StepIO<A>{p.x, p.old, p.out, p.ldx, p.ldo, p.ldout, p.a, p.b, p.s};
}

// A pointer read from device memory (a batch record, a pointer table) has no
// known address space, and its accesses become flat ones, which count as LDS
// accesses too: every wait for an LDS read then waits for the loads in flight
// as well.  All such pointers are to global memory.  (Frames of 24..40^3
// double: 15.8 -> 14.1 ms a filter; 112 units of 24^3 x 12 complex64: 4.17 ->
// 3.84 ms.)
template <class T>
__device__ __forceinline__ T *global_ptr(T *p)
{
    return (T *)(__attribute__((address_space(1))) T *)reinterpret_cast<unsigned long>(p);
}

// element i of a uniform base pointer, addressed by a 32-bit byte offset so
// the load can use a scalar base plus a vector offset
template <class T>
__device__ __forceinline__ T ld_at(const T *base, unsigned i)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + i * (unsigned)sizeof(T));
}
template <class T>
__device__ __forceinline__ void st_at(T *base, unsigned i, T v)
{
    *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + i * (unsigned)sizeof(T)) = v;
}

// XCD-aware work order: the hardware hands workgroups to the 8 XCDs round
// robin, so workgroup b runs on XCD b % 8; mapping it to work item
// (b % 8) * per + b / 8 gives each XCD a contiguous range of work items.
__device__ __forceinline__ int xcd_work_item()
{
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

// The operator of a non-orthogonal cell, factored: D2_a[k] = beta_a w2[k],
// mixed c_ab[k] = alpha_ab w1[k], D1_a[k] = w1[k] / h_a.
template <class A>
struct NonorthArgs {
    StepArgs<A> b;
    A w1[kMaxR + 1];
    A w2[kMaxR + 1];
    A beta[3];
    A axy_hy;            // alpha_xy / h_y
    A axz, ayz;          // alpha_xz, alpha_yz
    A ihz;               // 1 / h_z
};

// The operator part of the kernel arguments of a grid (buffers, launch shape
// and step scalars are the caller's).
template <class A>
NonorthArgs<A> operator_args(const StencilGeom &g)
{
    NonorthArgs<A> q{};
    StepArgs<A> &p = q.b;
    p.nx = g.nx; p.ny = g.ny; p.nz = g.nz;
    for (int ax = 0; ax < 3; ++ax) {
        for (int k = 0; k <= kMaxR; ++k) p.c[ax][k] = (A)g.c[ax][k];
        for (int sd = 0; sd < 2; ++sd)
            for (int k = 0; k < 2; ++k) p.ph[ax][sd][k] = (A)g.phase[ax][sd][k];
        q.beta[ax] = (A)g.beta[ax];
    }
    for (int k = 0; k <= kMaxR; ++k) {
        q.w1[k] = (A)g.w1[k];
        q.w2[k] = (A)g.w2[k];
    }
    q.axy_hy = (A)(g.alpha[0] / g.h[1]);
    q.axz = (A)g.alpha[1];
    q.ayz = (A)g.alpha[2];
    q.ihz = (A)(1.0 / g.h[2]);
    return q;
}

// a run of VW consecutive x points, loaded and stored as one vector
template <class S, int VW>
struct alignas(sizeof(S) * VW) VRun {
    S v[VW];
};

template <class S, int VW>
__device__ __forceinline__ VRun<S, VW> vzero()
{
    VRun<S, VW> r;
#pragma unroll
    for (int e = 0; e < VW; ++e) r.v[e] = S(0);
    return r;
}

template <int VW, class S>
__device__ __forceinline__ VRun<S, VW> vld(const S *base, unsigned i)
{
    return *reinterpret_cast<const VRun<S, VW> *>(reinterpret_cast<const char *>(base) + i * (unsigned)sizeof(S));
}

// A run of storage type T as it was loaded, and its values in compute type S.
// bfloat16 pairs stay packed until they are used: unpacked at the load, the
// values would wait for memory where the loads are issued, a plane too early.
template <class S, class T, int VW>
struct Held {
    VRun<S, VW> r;
    __device__ __forceinline__ VRun<S, VW> get() const { return r; }
};
template <int VW>
struct alignas(2 * VW) Held<float, bf16, VW> {
    unsigned w[VW / 2];
    __device__ __forceinline__ VRun<float, VW> get() const
    {
        VRun<float, VW> r;
#pragma unroll
        for (int e = 0; e < VW; ++e)
            r.v[e] = __uint_as_float(e & 1 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16);
        return r;
    }
};
template <int VW, class S, class T>
__device__ __forceinline__ Held<S, T, VW> vldh(const T *base, unsigned i)
{
    return *reinterpret_cast<const Held<S, T, VW> *>(reinterpret_cast<const char *>(base) + i * (unsigned)sizeof(T));
}
// a run stored back as T
template <int VW, class S, class T>
__device__ __forceinline__ void vstc(T *base, unsigned i, const VRun<S, VW> &v)
{
    VRun<T, VW> t;
#pragma unroll
    for (int e = 0; e < VW; ++e) t.v[e] = StoreAs<T>::from(v.v[e]);
    *reinterpret_cast<VRun<T, VW> *>(reinterpret_cast<char *>(base) + i * (unsigned)sizeof(T)) = t;
}

template <class A>
struct NlArgs {
    const int *atom_pt_off, *pt_gpos, *pt_img, *pt_atom, *cov_off, *cov_gpos, *ent_pt;
    const A *chi, *gamma, *phase;
    int n_atom, n_cov, npm;
};

template <class A>
__device__ __forceinline__ NlArgs<A> global_args(const NlArgs<A> &p)
{
    return NlArgs<A>{global_ptr(p.atom_pt_off), global_ptr(p.pt_gpos), global_ptr(p.pt_img), global_ptr(p.pt_atom),
                     global_ptr(p.cov_off), global_ptr(p.cov_gpos), global_ptr(p.ent_pt), global_ptr(p.chi),
                     global_ptr(p.gamma), global_ptr(p.phase), p.n_atom, p.n_cov, p.npm};
}

// One unit of a batch.
template <class A>
struct BatchRec {
    NonorthArgs<A> q;           // operator of the unit; pointers and a, b, s set per step
    const void *buf[4];         // X, D1, D2, none
    long ld[4];
    int item0;                  // first stencil work item
    int g_item0, s_item0;       // first gather / scatter block
    int ncol;
    int s_cpw;                  // scatter columns per wave
    long beta_off;              // first beta element of the unit
    NlArgs<A> nl;
    // gather by parts (units with large spheres): sphere point ranges
    // [pb, pe) of at most kGatherPartPts points of one atom, the first part
    // of each atom (n_atom + 1), and the unit's first partial sum
    const int2 *parts;
    const int *atom_part;
    int nparts;
    int r_item0;                // first reduction block
    long part_off;
};


}  // namespace
}  // namespace gpu
}  // namespace lynx
