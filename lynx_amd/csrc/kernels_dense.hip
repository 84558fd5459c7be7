// Dense kernels for narrow FP64 / complex128 blocks (up to kNarrowReal real
// or kNarrowComplex complex columns), one launch for any number of units of
// equal shape: the Hermitian Gram product and the rotation of a block on the
// FP64 matrix cores, and the n x n Cholesky inverse and eigensolve, one
// workgroup per matrix with the matrix in LDS.
#include "kernels.hpp"
#include "common.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

namespace lynx {
namespace gpu {
namespace {

typedef double double4v __attribute__((ext_vector_type(4)));

// block u of a batch: entry u of a device pointer table, or the one block
template <class S>
__device__ __forceinline__ S *unit_of(const NarrowBlocks &b, int u)
{
    // (the address space of a pointer read from memory is not known otherwise)
    typedef __attribute__((address_space(1))) S *G;
    return (S *)(G)reinterpret_cast<unsigned long>(b.table ? b.table[u] : b.base);
}

// -------------------------------------------------------------------- Gram --
// Partial products of S = A^H B (upper 16 x 16 tiles; B is A for the overlap,
// H A for the projection, whose Hermitian part is taken) over one chunk of
// rows, on v_mfma_f64_16x16x4f64 straight from memory.  Lane l holds column
// l % 16 of a tile and rows 4 (l / 16) .. + 3 of each 16-row step (two
// complex rows of an 8-row step), 32 contiguous bytes, so a wave reads whole
// 128-byte lines of 16 columns and its four values are four k slices of the
// product (the order of the k index is the same for both operands).  Complex
// columns count as real columns of twice the length: the real part is the
// product with B as stored, the imaginary part the one with (b_i, -b_r).
// Bound by the read of the block (HBM or L2): 112 units of 13,824 x 12
// complex (297 MB) take 110 us for the overlap and 173 us for the projection
// (3.4 TB/s of two blocks), where a batched GEMM, which pads the n x n output
// to 32 x 32 and leaves K in one workgroup, takes 1690 us; 27,000 x 24 real
// takes 8 and 11 us, in few waves.
template <bool CPLX, int T, bool SAME>
__global__ void __launch_bounds__(256) k_narrow_gram(NarrowBlocks a, long lda, NarrowBlocks b, long ldb, long K,
                                                     int n, long kch, int vec, double *__restrict__ part)
{
    constexpr int NT = T * (T + 1) / 2, CW = CPLX ? 2 : 1;
    const int u = blockIdx.y;
    const double *A = unit_of<double>(a, u), *B = SAME ? A : unit_of<double>(b, u);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int lr = l & 15, lk = l >> 4;
    const long len = K * CW;                                   // column length in doubles
    const long beg = (long)blockIdx.x * kch * CW, end = min(len, beg + kch * CW);
    long ca[T], cb[T];
    bool cv[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int c = 16 * t + lr;
        cv[t] = c < n;
        ca[t] = (long)(cv[t] ? c : 0) * lda * CW;
        cb[t] = (long)(cv[t] ? c : 0) * ldb * CW;
    }
    auto load = [&](const double *X, long col, long r, bool ok) {
        double4v v = double4v{0.0, 0.0, 0.0, 0.0};
        const double *p = X + col + r;
        if (r + 3 < end) {
            if (vec) {
                const double2 x = reinterpret_cast<const double2 *>(p)[0], y = reinterpret_cast<const double2 *>(p)[1];
                v = double4v{x.x, x.y, y.x, y.y};
            } else {
                v = double4v{p[0], p[1], p[2], p[3]};
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (r + i < end) v[i] = p[i];
        }
        if (!ok) v = double4v{0.0, 0.0, 0.0, 0.0};
        return v;
    };
    double4v re[NT], im[CPLX ? NT : 1];
#pragma unroll
    for (int t = 0; t < NT; ++t) re[t] = double4v{0.0, 0.0, 0.0, 0.0};
    if constexpr (CPLX) {
#pragma unroll
        for (int t = 0; t < NT; ++t) im[t] = double4v{0.0, 0.0, 0.0, 0.0};
    }
    for (long r0 = beg + 16 * w; r0 < end; r0 += 64) {
        const long r = r0 + 4 * lk;
        double4v x[T], y[T];
#pragma unroll
        for (int t = 0; t < T; ++t) x[t] = load(A, ca[t], r, cv[t]);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if constexpr (SAME) y[t] = x[t];
            else y[t] = load(B, cb[t], r, cv[t]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            int q = 0;
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = i; j < T; ++j, ++q) {
                    re[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][s], y[j][s], re[q], 0, 0, 0);
                    if constexpr (CPLX)
                        im[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][s], s % 2 ? -y[j][s - 1] : y[j][s + 1],
                                                                     im[q], 0, 0, 0);
                }
        }
    }
    // the four waves' sums in a fixed order, then the tiles as they lie in
    // the registers: [tile][re | im][lane][4]
    __shared__ double4v red[NT * CW * 64];
    for (int k = 0; k < 4; ++k) {
        if (w == k) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                double4v *d = red + t * CW * 64 + l;
                d[0] = k ? d[0] + re[t] : re[t];
                if constexpr (CPLX) d[64] = k ? d[64] + im[t] : im[t];
            }
        }
        __syncthreads();
    }
    double4v *P = reinterpret_cast<double4v *>(part) + ((long)u * gridDim.x + blockIdx.x) * (NT * CW * 64);
    for (int i = threadIdx.x; i < NT * CW * 64; i += 256) P[i] = red[i];
}

// S (n x n per unit) = alpha * the sum of the chunks' partial tiles, in chunk
// order, with the upper triangle mirrored and a real diagonal.  One thread
// per stored tile value: a single n = 24 product has 768 of them with 128
// partials each (12 us, a chain of L2 loads; 100 us with one thread per
// output of the general sum).
template <bool CPLX>
__global__ void __launch_bounds__(64) k_narrow_gram_sum(const double *__restrict__ part, int nchunk, int T, int n,
                                                        double alpha, double *__restrict__ C)
{
    constexpr int CW = CPLX ? 2 : 1;
    const int u = blockIdx.y, per = T * (T + 1) / 2 * CW * 256;
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= per) return;
    const double *P = part + (long)u * nchunk * per + i;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int c = 0;
    for (; c + 3 < nchunk; c += 4) {
        s0 += P[(long)c * per];
        s1 += P[(long)(c + 1) * per];
        s2 += P[(long)(c + 2) * per];
        s3 += P[(long)(c + 3) * per];
    }
    for (; c < nchunk; ++c) s0 += P[(long)c * per];
    const double v = alpha * ((s0 + s1) + (s2 + s3));
    const int reg = i & 3, lane = (i >> 2) & 63, t = i / (CW * 256);
    const bool imag = CPLX && ((i >> 8) & 1);
    int ti = 0, q = t;
    while (q >= T - ti) q -= T - ti++;
    const int row = 16 * ti + (lane >> 4) + 4 * reg, col = 16 * (ti + q) + (lane & 15);
    if (col >= n || row > col) return;
    double *M = C + (long)u * n * n * CW;
    M[(row + (long)col * n) * CW + imag] = imag && row == col ? 0.0 : v;
    if (row != col) M[(col + (long)row * n) * CW + imag] = imag ? -v : v;
}

// ---------------------------------------------------------------- rotation --
// C = A Q for n columns (C may be A: a wave holds its 16 rows of every column
// before it writes).  The product is formed as C^T = Q^T A^T, so that a lane
// holds one row and four columns of each output tile and a store covers 16
// consecutive rows of a column.  Q sits in LDS, padded with zeros to whole
// 16-column tiles.  Bound by the read and write of the block: 96 us for 112
// units of 13,824 x 12 complex in place (6.2 TB/s, a part of it from the last
// level cache) where the batched GEMM takes 256 us into another block and the
// copy back as long again; 7 us for 27,000 x 24 real (the GEMM: 14 us).
template <bool CPLX, int T>
__global__ void __launch_bounds__(256) k_narrow_rotate(NarrowBlocks a, long lda, NarrowBlocks c, long ldc, long K,
                                                       int n, const double *__restrict__ Q)
{
    constexpr int CW = CPLX ? 2 : 1, NP = 16 * T, PQ = NP + 1;
    __shared__ double sq[NP * PQ * CW];                        // [re | im][j][k], pitch PQ
    const int u = blockIdx.y;
    Q += (long)u * n * n * CW;
    for (int i = threadIdx.x; i < NP * NP; i += 256) {
        const int k = i % NP, j = i / NP;
        const bool in = k < n && j < n;
#pragma unroll
        for (int p = 0; p < CW; ++p) sq[p * NP * PQ + j * PQ + k] = in ? Q[((long)j * n + k) * CW + p] : 0.0;
    }
    __syncthreads();
    const double *A = unit_of<double>(a, u);
    double *C = unit_of<double>(c, u);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int lr = l & 15, lk = l >> 4;
    const long step = (long)gridDim.x * 64;
    for (long r0 = (long)blockIdx.x * 64 + 16 * w; r0 < K; r0 += step) {
        const long r = r0 + lr;
        const bool rv = r < K;
        double x[4 * T][CW];
#pragma unroll
        for (int s = 0; s < 4 * T; ++s) {
            const int k = 4 * s + lk;
            const bool in = rv && k < n;
            const double *p = A + (in ? (r + (long)k * lda) * CW : 0);
#pragma unroll
            for (int z = 0; z < CW; ++z) x[s][z] = in ? p[z] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            double4v re = double4v{0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll
            for (int s = 0; s < 4 * T; ++s) {
                const double *q = sq + (16 * t + lr) * PQ + 4 * s + lk;
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(q[0], x[s][0], re, 0, 0, 0);
                if constexpr (CPLX) {
                    const double qi = q[NP * PQ];
                    im = __builtin_amdgcn_mfma_f64_16x16x4f64(q[0], x[s][1], im, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-qi, x[s][1], re, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f64_16x16x4f64(qi, x[s][0], im, 0, 0, 0);
                }
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = 16 * t + lk + 4 * v;
                if (rv && j < n) {
                    if constexpr (CPLX)
                        reinterpret_cast<double2 *>(C)[r + (long)j * ldc] = make_double2(re[v], im[v]);
                    else
                        C[r + (long)j * ldc] = re[v];
                }
            }
        }
    }
}

// ----------------------------------------------------- small n x n matrices --
struct Cx {
    double re, im;
};
__device__ __forceinline__ double conj_(double a) { return a; }
__device__ __forceinline__ Cx conj_(Cx a) { return {a.re, -a.im}; }
__device__ __forceinline__ double mul(double a, double b) { return a * b; }
__device__ __forceinline__ Cx mul(Cx a, Cx b) { return {fma(a.re, b.re, -a.im * b.im), fma(a.re, b.im, a.im * b.re)}; }
__device__ __forceinline__ Cx mul(double a, Cx b) { return {a * b.re, a * b.im}; }
__device__ __forceinline__ double sub(double a, double b) { return a - b; }
__device__ __forceinline__ Cx sub(Cx a, Cx b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ double add(double a, double b) { return a + b; }
__device__ __forceinline__ Cx add(Cx a, Cx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ double real_(double a) { return a; }
__device__ __forceinline__ double real_(Cx a) { return a.re; }
__device__ __forceinline__ double abs_(double a) { return fabs(a); }
__device__ __forceinline__ double abs_(Cx a) { return hypot(a.re, a.im); }
__device__ __forceinline__ double peak(double a) { return fabs(a); }           // largest component, NaN of a NaN
__device__ __forceinline__ double peak(Cx a)
{
    return isnan(a.re) || isnan(a.im) ? a.re + a.im : fmax(fabs(a.re), fabs(a.im));
}
__device__ __forceinline__ double scale2(double a, int e) { return ldexp(a, e); }
__device__ __forceinline__ Cx scale2(Cx a, int e) { return {ldexp(a.re, e), ldexp(a.im, e)}; }
__device__ __forceinline__ double norm2(double a) { return a * a; }
__device__ __forceinline__ double norm2(Cx a) { return fma(a.re, a.re, a.im * a.im); }
template <class E> __device__ __forceinline__ E from_real(double a);
template <> __device__ __forceinline__ double from_real<double>(double a) { return a; }
template <> __device__ __forceinline__ Cx from_real<Cx>(double a) { return {a, 0.0}; }

// S = R^H R (R upper triangular), S replaced by R^-1 (zeros below).  Step k
// of the factorisation and of the inverse go together: with row k of R known,
// the trailing part of S loses its outer product and, W holding I times the
// inverses of the eliminated columns, column j > k of W loses R(k, j) times
// column k of R^-1.  Three barriers a step; info is the order of the first
// pivot that is not positive (0: none), as LAPACK's potrf has it.  Bound by
// the barriers: 22 us at n = 24 real, 10 us for 112 matrices of n = 12
// complex (potrf and trtri: 64 us in two calls, 29 us).
template <class E>
__global__ void __launch_bounds__(256) k_narrow_cholesky(double *__restrict__ M, int n, int *__restrict__ info)
{
    extern __shared__ __align__(16) unsigned char smem[];
    E *S = reinterpret_cast<E *>(smem), *W = S + n * (n + 1);  // column-major, pitch n + 1
    const int P = n + 1, t = threadIdx.x, u = blockIdx.x;
    E *G = reinterpret_cast<E *>(M) + (long)u * n * n;
    for (int i = t; i < n * n; i += 256) {
        const int r = i % n, c = i / n;
        S[r + c * P] = G[i];
        W[r + c * P] = from_real<E>(r == c ? 1.0 : 0.0);
    }
    __syncthreads();
    int bad = 0;
    for (int k = 0; k < n; ++k) {
        const double d = real_(S[k + k * P]);
        if (!(d > 0.0)) {
            bad = k + 1;
            break;
        }
        const double inv = 1.0 / sqrt(d);
        __syncthreads();
        for (int i = t; i < n; i += 256) {
            if (i > k) S[k + i * P] = mul(inv, S[k + i * P]);   // row k of R
            else W[i + k * P] = mul(inv, W[i + k * P]);         // column k of R^-1
        }
        __syncthreads();
        const int m = n - 1 - k;                                // trailing columns
        for (int i = t; i < m * n; i += 256) {
            const int c = k + 1 + i / n, r = i % n;
            const E f = S[k + c * P];
            if (r <= k) W[r + c * P] = sub(W[r + c * P], mul(f, W[r + k * P]));
            else if (r <= c) S[r + c * P] = sub(S[r + c * P], mul(conj_(S[k + r * P]), f));
        }
        __syncthreads();
    }
    if (t == 0) info[u] = bad;
    if (bad) return;
    for (int i = t; i < n * n; i += 256) {
        const int r = i % n, c = i / n;
        G[i] = r <= c ? W[r + c * P] : from_real<E>(0.0);
    }
}

// Eigenvectors (replacing H) and ascending eigenvalues of a Hermitian n x n
// matrix by cyclic Jacobi rotations, n / 2 disjoint pairs at a time in
// round-robin order: a thread rotates the 2 x 2 block of two pairs of A, or
// two entries of a row of V.  A pass over all pairs is n - 1 rounds of two
// barriers; the passes end when no off-diagonal entry met in one exceeded
// 2^-53 of the Frobenius norm (the backward error of a tridiagonal
// eigensolver).  The projected matrix of a converging subspace is nearly
// diagonal, which a Jacobi pass exploits and the reduction to tridiagonal
// form does not, and one workgroup with the matrix in LDS replaces about 100
// launches of the blocked algorithm, each a few microseconds for these n:
// 167 us at n = 24 real against 560 us of kernels and 600 us of gaps between
// them, 82 us for 112 matrices of n = 12 complex against 1600 us.  Bound by
// LDS latency, two dependent accesses and two barriers a round.
template <class E, int NT>
__global__ void __launch_bounds__(NT) k_narrow_eig(double *__restrict__ M, int n, double *__restrict__ eval,
                                                   int *__restrict__ info)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int m = (n + 1) & ~1, h = m / 2, P = m + 1;
    E *A = reinterpret_cast<E *>(smem), *V = A + m * P, *sn = V + m * P;    // sn: sine times the phase
    double *cs = reinterpret_cast<double *>(sn + h), *ta = cs + h;          // cosine, tangent times |a_pq|
    double *mx = ta + h, *ev = mx + h;                                      // largest |a_pq| met, diagonal
    const int t = threadIdx.x, u = blockIdx.x;
    E *G = reinterpret_cast<E *>(M) + (long)u * n * n;
    double s = 0.0;
    for (int i = t; i < m * m; i += NT) {
        const int r = i % m, c = i / m;
        E v = from_real<E>(0.0);
        if (r < n && c < n) {
            v = r <= c ? G[r + (long)c * n] : conj_(G[c + (long)r * n]);
            if (r == c) v = from_real<E>(real_(v));
        }
        A[r + c * P] = v;
        V[r + c * P] = from_real<E>(r == c ? 1.0 : 0.0);
        s += norm2(v);
    }
    __shared__ double red[NT / 64];
    auto over_threads = [&](double v, auto op) {               // over the workgroup, all threads get it
        for (int o = 32; o; o >>= 1) v = op(v, __shfl_xor(v, o));
        __syncthreads();
        if ((t & 63) == 0) red[t >> 6] = v;
        __syncthreads();
        v = red[0];
        for (int i = 1; i < NT / 64; ++i) v = op(v, red[i]);
        return v;
    };
    auto plus = [](double a, double b) { return a + b; };
    s = over_threads(s, plus);
    // Squares out of range: the matrix is scaled by a power of two, or, with a
    // value that is no number or infinite, refused (a NaN would pass every
    // test below as converged)
    int e = 0;
    if (!(s <= 0x1p900) || s < 0x1p-900) {
        double a = 0.0;
        for (int i = t; i < m * m; i += NT) {
            const double v = peak(A[i % m + i / m * P]);
            a = v <= 0x1.fffffffffffffp1023 ? fmax(a, v) : HUGE_VAL;
            if (a == HUGE_VAL) break;
        }
        a = over_threads(a, [](double x, double y) { return fmax(x, y); });
        if (a == HUGE_VAL) {
            if (t == 0) info[u] = 1;
            return;
        }
        e = a > 0.0 ? ilogb(a) : 0;
        s = 0.0;
        for (int i = t; i < m * m; i += NT) {
            E &v = A[i % m + i / m * P];
            v = scale2(v, -e);
            s += norm2(v);
        }
        s = over_threads(s, plus);
    }
    const double tol = sqrt(s) * 0x1p-53;
    double big = 0.0;
    bool done = false;
    auto pair = [&](int k, int round, int &p, int &q) {
        int x = k ? round + k : round, y = k ? round - k : m - 1;
        if (x >= m - 1 && k) x -= m - 1;
        if (y < 0) y += m - 1;
        p = min(x, y);
        q = max(x, y);
    };
    const int blocks = h * (h + 1) / 2;
    for (int pass = 0; pass < 40 && !done; ++pass) {
        big = 0.0;
        for (int round = 0; round < m - 1; ++round) {
            if (t < h) {
                int p, q;
                pair(t, round, p, q);
                const E c = A[p + q * P];
                const double ac = abs_(c);
                big = fmax(big, ac);
                double co = 1.0, tn = 0.0;
                E si = from_real<E>(0.0);
                if (ac > 0.0) {
                    const double tau = (real_(A[q + q * P]) - real_(A[p + p * P])) / (2.0 * ac);
                    const double tt = copysign(1.0, tau) / (fabs(tau) + sqrt(fma(tau, tau, 1.0)));
                    co = 1.0 / sqrt(fma(tt, tt, 1.0));
                    si = mul(tt * co / ac, c);
                    tn = tt * ac;
                }
                cs[t] = co;
                sn[t] = si;
                ta[t] = tn;
            }
            __syncthreads();
            for (int i = t; i < blocks + m * h; i += NT) {
                if (i < blocks) {
                    // block (a, b), a <= b, of the upper triangle of pairs
                    int b = (int)((sqrtf(8.0f * i + 1.0f) - 1.0f) * 0.5f);
                    while ((b + 1) * (b + 2) / 2 <= i) ++b;
                    while (b * (b + 1) / 2 > i) --b;
                    const int a = i - b * (b + 1) / 2;
                    int p, q, x, y;
                    pair(a, round, p, q);
                    if (a == b) {
                        A[p + p * P] = from_real<E>(real_(A[p + p * P]) - ta[a]);
                        A[q + q * P] = from_real<E>(real_(A[q + q * P]) + ta[a]);
                        if (cs[a] != 1.0 || ta[a] != 0.0) A[p + q * P] = A[q + p * P] = from_real<E>(0.0);
                        continue;
                    }
                    pair(b, round, x, y);
                    const E px = A[p + x * P], py = A[p + y * P], qx = A[q + x * P], qy = A[q + y * P];
                    // columns x, y by the pair b, then rows p, q by the pair a
                    const E sb = sn[b], sa = sn[a];
                    const double cb = cs[b], ca = cs[a];
                    const E p1 = sub(mul(cb, px), mul(conj_(sb), py)), p2 = add(mul(sb, px), mul(cb, py));
                    const E q1 = sub(mul(cb, qx), mul(conj_(sb), qy)), q2 = add(mul(sb, qx), mul(cb, qy));
                    const E r1 = sub(mul(ca, p1), mul(sa, q1)), r2 = sub(mul(ca, p2), mul(sa, q2));
                    const E s1 = add(mul(conj_(sa), p1), mul(ca, q1)), s2 = add(mul(conj_(sa), p2), mul(ca, q2));
                    A[p + x * P] = r1;
                    A[x + p * P] = conj_(r1);
                    A[p + y * P] = r2;
                    A[y + p * P] = conj_(r2);
                    A[q + x * P] = s1;
                    A[x + q * P] = conj_(s1);
                    A[q + y * P] = s2;
                    A[y + q * P] = conj_(s2);
                } else {
                    const int r = (i - blocks) % m, a = (i - blocks) / m;
                    int p, q;
                    pair(a, round, p, q);
                    const E vp = V[r + p * P], vq = V[r + q * P], sa = sn[a];
                    const double ca = cs[a];
                    V[r + p * P] = sub(mul(ca, vp), mul(conj_(sa), vq));
                    V[r + q * P] = add(mul(sa, vp), mul(ca, vq));
                }
            }
            __syncthreads();
        }
        if (t < h) mx[t] = big;
        __syncthreads();
        double all = 0.0;
        for (int i = 0; i < h; ++i) all = fmax(all, mx[i]);
        done = !(all > tol);
        __syncthreads();
    }
    for (int i = t; i < n; i += NT) ev[i] = real_(A[i + i * P]);
    __syncthreads();
    // ascending order (ties by index)
    for (int i = t; i < n * n; i += NT) {
        const int r = i % n, c = i / n;
        int rank = 0;
        for (int j = 0; j < n; ++j) rank += ev[j] < ev[c] || (ev[j] == ev[c] && j < c);
        G[r + (long)rank * n] = V[r + c * P];
        if (r == 0) eval[(long)u * n + rank] = ldexp(ev[c], e);
    }
    if (t == 0) info[u] = done ? 0 : 1;
}

void check_launch(const char *what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) fail(2, std::string(what) + ": " + hipGetErrorString(e));
}

template <class F>
void by_tiles(int T, F &&f)
{
    switch (T) {
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        default: f(std::integral_constant<int, 4>{}); break;
    }
}

// dynamic LDS of the matrix kernels
size_t cholesky_lds(bool cplx, int n) { return 2 * (size_t)n * (n + 1) * (cplx ? 16 : 8); }
size_t eig_lds(bool cplx, int n)
{
    const size_t m = (n + 1) & ~1, es = cplx ? 16 : 8;
    return 2 * m * (m + 1) * es + m / 2 * es + (3 * (m / 2) + n) * sizeof(double);
}

}  // namespace

bool narrow_fits(int e, int n)
{
    return n >= 1 && ((e == F64 && n <= kNarrowReal) || (e == C128 && n <= kNarrowComplex));
}

int narrow_gram_chunks(int units, long K)
{
    // about 512 workgroups in all, at least 64 rows (16 per wave) each
    const long most = std::max<long>(1, K / 64);
    return (int)std::max<long>(1, std::min({most, 128L, (512L + units - 1) / units}));
}

size_t narrow_gram_work(int e, int n, int units, long K)
{
    const int T = (n + 15) / 16;
    return (size_t)units * narrow_gram_chunks(units, K) * (T * (T + 1) / 2) * (e == C128 ? 512 : 256) * sizeof(double);
}

void narrow_gram(int e, const NarrowBlocks &A, long lda, const NarrowBlocks &B, long ldb, bool same, bool aligned,
                 long K, int n, int units, double alpha, void *C, void *work, hipStream_t st)
{
    const bool cplx = e == C128;
    const int T = (n + 15) / 16, nch = narrow_gram_chunks(units, K);
    // chunks of whole 16-row steps of the four waves
    const long kch = ((K + nch - 1) / nch + 63) / 64 * 64;
    // 16-byte loads of two doubles (complex values are 16-byte aligned)
    const int vec = aligned && (cplx || (lda % 2 == 0 && ldb % 2 == 0));
    double *part = static_cast<double *>(work);
    auto go = [&](auto cx, auto tt, auto sm) {
        k_narrow_gram<decltype(cx)::value, decltype(tt)::value, decltype(sm)::value>
            <<<dim3(nch, units), 256, 0, st>>>(A, lda, B, ldb, K, n, kch, vec, part);
    };
    by_tiles(T, [&](auto tt) {
        using Y = std::true_type;
        using N = std::false_type;
        if constexpr (decltype(tt)::value <= kNarrowComplex / 16) {
            if (cplx) {
                if (same) go(Y{}, tt, Y{});
                else go(Y{}, tt, N{});
                return;
            }
        }
        if (same) go(N{}, tt, Y{});
        else go(N{}, tt, N{});
    });
    check_launch("k_narrow_gram");
    const int per = T * (T + 1) / 2 * (cplx ? 512 : 256);
    if (cplx) k_narrow_gram_sum<true><<<dim3(per / 64, units), 64, 0, st>>>(part, nch, T, n, alpha, (double *)C);
    else k_narrow_gram_sum<false><<<dim3(per / 64, units), 64, 0, st>>>(part, nch, T, n, alpha, (double *)C);
    check_launch("k_narrow_gram_sum");
}

void narrow_rotate(int e, const NarrowBlocks &A, long lda, const NarrowBlocks &C, long ldc, long K, int n, int units,
                   const void *Q, hipStream_t st)
{
    const int nb = (int)std::max<long>(1, std::min<long>((K + 63) / 64, (4096 + units - 1) / units));
    by_tiles((n + 15) / 16, [&](auto tt) {
        constexpr int T = decltype(tt)::value;
        if constexpr (T <= kNarrowComplex / 16) {
            if (e == C128) {
                k_narrow_rotate<true, T><<<dim3(nb, units), 256, 0, st>>>(A, lda, C, ldc, K, n, (const double *)Q);
                return;
            }
        }
        k_narrow_rotate<false, T><<<dim3(nb, units), 256, 0, st>>>(A, lda, C, ldc, K, n, (const double *)Q);
    });
    check_launch("k_narrow_rotate");
}

void narrow_cholesky_inverse(int e, void *S, int n, int units, int *info, hipStream_t st)
{
    const size_t lds = cholesky_lds(e == C128, n);
    if (e == C128) k_narrow_cholesky<Cx><<<units, 256, lds, st>>>((double *)S, n, info);
    else k_narrow_cholesky<double><<<units, 256, lds, st>>>((double *)S, n, info);
    check_launch("k_narrow_cholesky");
}

void narrow_eig(int e, void *H, int n, int units, double *eval, int *info, hipStream_t st)
{
    const size_t lds = eig_lds(e == C128, n);
    if (e == C128) {
        if (n <= 16) k_narrow_eig<Cx, 256><<<units, 256, lds, st>>>((double *)H, n, eval, info);
        else k_narrow_eig<Cx, 512><<<units, 512, lds, st>>>((double *)H, n, eval, info);
    } else {
        if (n <= 32) k_narrow_eig<double, 256><<<units, 256, lds, st>>>((double *)H, n, eval, info);
        else k_narrow_eig<double, 1024><<<units, 1024, lds, st>>>((double *)H, n, eval, info);
    }
    check_launch("k_narrow_eig");
}

}  // namespace gpu
}  // namespace lynx
