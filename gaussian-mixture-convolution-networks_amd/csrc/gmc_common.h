// Shared device helpers of libgmc_hip (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gmc_hip.h"

namespace gmc {

constexpr int kBlock = 256;          // threads per workgroup of the dense kernels (4 wavefronts)
constexpr int kWave = 64;

template <int D> struct Kappa;       // (2 pi)^(-D/2)
template <> struct Kappa<2> { static constexpr double v = 0.15915494309189535; };
template <> struct Kappa<3> { static constexpr double v = 0.06349363593424097; };

// 0.5 * log2(e): folded into the Cholesky factor so that the kernel's exponential is a bare exp2
constexpr double kHalfLog2e = 0.72134752044448170368;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// exp2 of a non-positive argument for the pair loops.  float: the hardware instruction.  double: 2^x = 2^e 2^(j/256) 2^r
// with x = e + j/256 + r, |r| <= 1/512: the integer 256 e + j comes out of the low mantissa bits of x * 256 + 1.5 * 2^52
// (round to nearest), 2^(j/256) from a table of 256 entries in LDS and 2^r from four FMAs (truncation error 4e-17;
// the result is within 2 ulp): 14 vector instructions, four fewer than the library routine (measured).
constexpr int kExp2Table = 256;
// The table of the calling workgroup (float kernels have none and spend no LDS on it); a barrier must lie between this
// call and the first pair_exp2.
template <typename T> __device__ __forceinline__ const T* exp2_table();
template <> __device__ __forceinline__ const float* exp2_table<float>() { return nullptr; }
template <> __device__ __forceinline__ const double* exp2_table<double>() {
    __shared__ double tab[kExp2Table];
    for (int i = threadIdx.x; i < kExp2Table; i += blockDim.x) tab[i] = exp2(double(i) * (1.0 / kExp2Table));
    return tab;
}
// Issue of a wavefront's exponentials and cross-lane instructions in one go.  The SIMD issues FP32 additions, products and
// FMAs of two wavefronts side by side (2.2 - 2.8 cycles each, two or more wavefronts); exponentials, DPP, permlane and
// conversion instructions go alone, and one that meets the FP32 stream of the other wavefronts stops that pairing for longer
// than it takes itself.  At a raised wave priority a wavefront issues a batch of them back to back.  Measured, cycles (of
// 2.4 GHz, wall time) that eight of them add to 96 FMAs, four wavefronts per SIMD, without / with the priority: v_exp_f32
// 14.2 / 8.1, DPP addition 15 / 3, permlane swap 17.6 / 7.6, v_cvt_pk_bf16_f32 13.5 / 4.3; v_cndmask, v_and and compares
// 2 - 4 either way, matrix instructions 13 either way.  The arguments pin the values: what is computed between the calls
// stays between them.
template <int N>
__device__ __forceinline__ void slow_issue_begin(const float (&v)[N], int n = N) {
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (i < n) asm volatile("" :: "v"(v[i]));
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(3);
}
template <int N>
__device__ __forceinline__ void slow_issue_end(float (&v)[N], int n = N) {
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (i < n) asm volatile("" : "+v"(v[i]));
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ float pair_exp2(float x, const float*) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ double pair_exp2(double x, const double* __restrict__ tab) {
    constexpr double kMagic = 6755399441055744.0;                       // 1.5 * 2^52
    // 2^x is 0 from -1075 on: below -1100 the high word becomes that of -1100.0 (the low word may stay), which keeps
    // the integer within 32 bits; a NaN compares false and stays one
    x = __hiloint2double(x < -1100.0 ? int(0xC0913000u) : __double2hiint(x), __double2loint(x));
    const double t = __builtin_fma(x, double(kExp2Table), kMagic);
    const int k = __double2loint(t);                                    // 256 e + j, two's complement
    const double r = __builtin_fma(t - kMagic, -1.0 / kExp2Table, x);
    double p = 9.6181291076284772e-3;                                   // ln2^4 / 24
    p = __builtin_fma(p, r, 5.5504108664821580e-2);                     // ln2^3 / 6
    p = __builtin_fma(p, r, 2.4022650695910071e-1);                     // ln2^2 / 2
    p = __builtin_fma(p, r, 6.9314718055994531e-1);                     // ln2
    p = __builtin_fma(p, r, 1.0);
    return ldexp(tab[k & (kExp2Table - 1)] * p, k >> 8);
}
// exp2 of the negated values of the first n of N pairs at once
template <int N>
__device__ __forceinline__ void pair_exp2_batch(const float (&q)[N], float (&e)[N], int n = N) {
    slow_issue_begin(q, n);
#pragma unroll
    for (int p = 0; p < N; ++p)
        if (p < n) e[p] = __builtin_amdgcn_exp2f(-q[p]);
    slow_issue_end(e, n);
}
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Reciprocals, quotients and roots of the per-Gaussian preparation, in double.  For float32 tensors they come from the
// hardware's estimates (v_rcp_f64 / v_rsq_f64, at least 2^-23), one third-order correction and, for quotients and roots, the
// remainder against the rounded result: correctly rounded but for cases within 2^-20 of an ulp of a tie, instead of about
// 15 instructions for a double division and 20 for a square root, which the staging of a Gaussian needs five to fifteen of.
// (The factor's a11 - u01^2 of a singular matrix is then what it is with the full sequences: without the remainders a
// matrix of ones came out as NaN.)  A float's entries keep every intermediate far inside double's range, so the scaling of
// the full sequences has nothing to do; zeros and infinities take the estimate, which is exact there, and roots of negative
// arguments give NaN.  float64 tensors use the compiler's sequences.  Values and gradients of 1200 mixtures of 60 Gaussians
// at 700 points are the same bit for bit as with the full sequences (2-D and 3-D, both forms).  Measured with those for float32 too / now, covariance
// form: 1600 mixtures of 5120 Gaussians at 100 points in 3-D forward 341 / 312 us (every Gaussian meets few points),
// 4000 of 64 at 64 points in 3-D backward 66.4 / 61.8 us, 800 of 10 at 784 points in 2-D 14.5 / 13.8 us; where a Gaussian
// meets many points 0 to 2 % (84 of 4644 at 755 points in 2-D backward 241 / 239 us).
template <typename T> __device__ __forceinline__ double reciprocal(double x);
template <> __device__ __forceinline__ double reciprocal<double>(double x) { return 1.0 / x; }
template <> __device__ __forceinline__ double reciprocal<float>(double x) {
    constexpr int kZeroOrInfinity = 0x264;
    const double r = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_amdgcn_class(x, kZeroOrInfinity) ? r : __builtin_fma(r, __builtin_fma(e, e, e), r);
}
// a / x with r = reciprocal<T>(x), x neither 0 nor infinite
__device__ __forceinline__ double quotient_of_reciprocal(double a, double x, double r) {
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-q, x, a), r, q);
}
struct Root { double value, inverse; bool special; };       // sqrt(x); float only: 1 / sqrt(x), x is 0 or infinite
template <typename T> __device__ __forceinline__ Root root(double x);
template <> __device__ __forceinline__ Root root<double>(double x) { return {sqrt(x), 0.0, false}; }
template <> __device__ __forceinline__ Root root<float>(double x) {
    constexpr int kZeroOrPositiveInfinity = 0x260;
    const double y = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y), y, 1.0);
    const double inv = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
    const double s = x * inv;
    const double value = __builtin_fma(__builtin_fma(-s, s, x), 0.5 * inv, s);
    const bool special = __builtin_amdgcn_class(x, kZeroOrPositiveInfinity);
    return {special ? x : value, special ? y : inv, special};
}
// a / r.value
template <typename T> __device__ __forceinline__ double over(double a, const Root& r) {
    if constexpr (sizeof(T) == 8) return a / r.value;
    const double q = a * r.inverse;
    return r.special ? q : __builtin_fma(__builtin_fma(-q, r.value, a), r.inverse, q);
}
// a / kHalfLog2e, rounded once for float64 tensors
template <typename T> __device__ __forceinline__ double over_half_log2e(double a) {
    if constexpr (sizeof(T) == 8) return a / kHalfLog2e; else return a * (1.0 / kHalfLog2e);
}

// Per-Gaussian quantities derived once from the stored record (weight, position b, inverse covariance C):
//   u     upper-triangular factor with u^T u = 0.5*log2(e) * sym(C)   (row-major packed: D=2: 00 01 11, D=3: 00 01 02 11 12 22)
//   nd    -(u * b)
//   bound max_i sum_j |u_ij b_j|: magnitude of the partial sums of (u x + nd) for every pair that matters
//   norm  (2 pi)^(-D/2) * sqrt(det C),  det of C as stored
// so that  exp(-1/2 (x-b)^T C (x-b)) = exp2(-|u x + nd|^2) = exp2(-|u (x - b)|^2).
template <int D> struct Derived {
    double u[D * (D + 1) / 2];
    double nd[D];
    double b[D];
    double bound;
    double norm;
    double w;
};

// `covariance_form`: the record stores the covariance; its inverse (transposed, as gm.evaluate packs it,
// src/gmc/mixture.py:149) is formed here in double, so the covariance-form API needs no separate inversion pass.
template <typename T, int D>
__device__ __forceinline__ void load_inverse_covariance(const T* __restrict__ c, bool covariance_form, double (&m)[D][D]) {
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) m[i][j] = double(c[i * D + j]);
    if (!covariance_form) return;
    if constexpr (D == 2) {
        const double det = m[0][0] * m[1][1] - m[0][1] * m[1][0];
        const double a = m[0][0], b = m[0][1], cc = m[1][0], d = m[1][1];
        // (S^-1)^T
        if constexpr (sizeof(T) == 4) {
            const double r = reciprocal<T>(det);
            if (r == 0.0 || det == 0.0) {
                m[0][0] = d * r; m[0][1] = -cc * r; m[1][0] = -b * r; m[1][1] = a * r;
            } else {
                m[0][0] = quotient_of_reciprocal(d, det, r); m[0][1] = -quotient_of_reciprocal(cc, det, r);
                m[1][0] = -quotient_of_reciprocal(b, det, r); m[1][1] = quotient_of_reciprocal(a, det, r);
            }
        } else {
            m[0][0] = d / det; m[0][1] = -cc / det; m[1][0] = -b / det; m[1][1] = a / det;
        }
    } else {
        double k[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int i1 = i == 0 ? 1 : 0, i2 = i == 2 ? 1 : 2;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int j1 = j == 0 ? 1 : 0, j2 = j == 2 ? 1 : 2;
                const double minor = m[i1][j1] * m[i2][j2] - m[i1][j2] * m[i2][j1];
                k[i][j] = ((i + j) & 1) ? -minor : minor;
            }
        }
        const double det = m[0][0] * k[0][0] + m[0][1] * k[0][1] + m[0][2] * k[0][2];
        // S^-1 = cofactor^T / det, hence (S^-1)^T = cofactor / det
        const double r = sizeof(T) == 4 ? reciprocal<T>(det) : 0.0;
        const bool plain = sizeof(T) == 4 && (r == 0.0 || det == 0.0);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                m[i][j] = sizeof(T) == 8 ? k[i][j] / det : plain ? k[i][j] * r : quotient_of_reciprocal(k[i][j], det, r);
    }
}

// Determinant of the D x D matrix of a Gaussian.  For float32 inputs the plain expansion in double is exact enough
// (its rounding error, up to a few thousand 2^-53 for condition numbers of several hundred, is far below 2^-24).  For
// float64 inputs the signed products of the expansion are formed and added as unevaluated pairs hi + lo (error-free
// product by FMA, error-free sum), so the result is the correctly rounded determinant of the stored entries also where
// the products cancel: once per Gaussian and workgroup, about a hundred instructions.
struct TwoDoubles { double hi, lo; };
__device__ __forceinline__ TwoDoubles exact_product(double a, double b) {
#pragma clang fp contract(off)
    const double p = a * b;
    return {p, __builtin_fma(a, b, -p)};
}
__device__ __forceinline__ TwoDoubles renormalised(double hi, double lo) {        // |hi| >= |lo|
#pragma clang fp contract(off)
    const double s = hi + lo;
    return {s, lo - (s - hi)};
}
__device__ __forceinline__ TwoDoubles times(TwoDoubles x, double c) {
#pragma clang fp contract(off)
    const double p = x.hi * c;
    const double e = __builtin_fma(x.lo, c, __builtin_fma(x.hi, c, -p));
    return renormalised(p, e);
}
__device__ __forceinline__ TwoDoubles plus(TwoDoubles x, TwoDoubles y) {
#pragma clang fp contract(off)
    const double s = x.hi + y.hi;
    const double v = s - x.hi;
    const double e = ((x.hi - (s - v)) + (y.hi - v)) + (x.lo + y.lo);
    return renormalised(s, e);
}
template <typename T, int D>
__device__ __forceinline__ double determinant(const double (&m)[D][D]) {
    if constexpr (sizeof(T) == 4) {
        if constexpr (D == 2) return m[0][0] * m[1][1] - m[0][1] * m[1][0];
        else return m[0][0] * (m[1][1] * m[2][2] - m[1][2] * m[2][1]) - m[0][1] * (m[1][0] * m[2][2] - m[1][2] * m[2][0]) +
                    m[0][2] * (m[1][0] * m[2][1] - m[1][1] * m[2][0]);
    } else if constexpr (D == 2) {
        const TwoDoubles d = plus(exact_product(m[0][0], m[1][1]), exact_product(-m[0][1], m[1][0]));
        return d.hi + d.lo;
    } else {
        TwoDoubles d = times(exact_product(m[0][0], m[1][1]), m[2][2]);
        d = plus(d, times(exact_product(-m[0][0], m[1][2]), m[2][1]));
        d = plus(d, times(exact_product(-m[0][1], m[1][0]), m[2][2]));
        d = plus(d, times(exact_product(m[0][1], m[1][2]), m[2][0]));
        d = plus(d, times(exact_product(m[0][2], m[1][0]), m[2][1]));
        d = plus(d, times(exact_product(-m[0][2], m[1][1]), m[2][0]));
        return d.hi + d.lo;
    }
}

// `cm` receives the inverse covariance
template <typename T, int D>
__device__ __forceinline__ Derived<D> derive(const T* __restrict__ g, bool covariance_form, double (&cm)[D][D]) {
    Derived<D> r;
    r.w = double(g[0]);
    load_inverse_covariance<T, D>(g + 1 + D, covariance_form, cm);
    if constexpr (D == 2) {
        const double c00 = cm[0][0], c01 = cm[0][1], c10 = cm[1][0], c11 = cm[1][1];
        const double det = determinant<T, 2>(cm);
        const double a00 = kHalfLog2e * c00, a01 = kHalfLog2e * 0.5 * (c01 + c10), a11 = kHalfLog2e * c11;
        const Root r0 = root<T>(a00);
        const double u00 = r0.value, u01 = over<T>(a01, r0);
        const double u11 = root<T>(a11 - u01 * u01).value;
        r.u[0] = u00; r.u[1] = u01; r.u[2] = u11;
        const double b0 = double(g[1]), b1 = double(g[2]);
        r.b[0] = b0; r.b[1] = b1;
        r.nd[0] = -(u00 * b0 + u01 * b1);
        r.nd[1] = -(u11 * b1);
        r.bound = fmax(fabs(u00 * b0) + fabs(u01 * b1), fabs(u11 * b1));
        r.norm = Kappa<2>::v * root<T>(det).value;
    } else {
        const double c00 = cm[0][0], c01 = cm[0][1], c02 = cm[0][2], c10 = cm[1][0], c11 = cm[1][1], c12 = cm[1][2],
                     c20 = cm[2][0], c21 = cm[2][1], c22 = cm[2][2];
        const double det = determinant<T, 3>(cm);
        const double a00 = kHalfLog2e * c00, a11 = kHalfLog2e * c11, a22 = kHalfLog2e * c22;
        const double a01 = kHalfLog2e * 0.5 * (c01 + c10), a02 = kHalfLog2e * 0.5 * (c02 + c20),
                     a12 = kHalfLog2e * 0.5 * (c12 + c21);
        const Root r0 = root<T>(a00);
        const double u00 = r0.value, u01 = over<T>(a01, r0), u02 = over<T>(a02, r0);
        const Root r1 = root<T>(a11 - u01 * u01);
        const double u11 = r1.value, u12 = over<T>(a12 - u01 * u02, r1);
        const double u22 = root<T>(a22 - u02 * u02 - u12 * u12).value;
        r.u[0] = u00; r.u[1] = u01; r.u[2] = u02; r.u[3] = u11; r.u[4] = u12; r.u[5] = u22;
        const double b0 = double(g[1]), b1 = double(g[2]), b2 = double(g[3]);
        r.b[0] = b0; r.b[1] = b1; r.b[2] = b2;
        r.nd[0] = -(u00 * b0 + u01 * b1 + u02 * b2);
        r.nd[1] = -(u11 * b1 + u12 * b2);
        r.nd[2] = -(u22 * b2);
        r.bound = fmax(fabs(u00 * b0) + fabs(u01 * b1) + fabs(u02 * b2), fmax(fabs(u11 * b1) + fabs(u12 * b2), fabs(u22 * b2)));
        r.norm = Kappa<3>::v * root<T>(det).value;
    }
    return r;
}

template <typename T, int D>
__device__ __forceinline__ Derived<D> derive(const T* __restrict__ g, bool covariance_form = false) {
    double cm[D][D];
    return derive<T, D>(g, covariance_form, cm);
}

// LDS record of one Gaussian for the pair loop: u, then nd ("shifted" form) or b ("centred" form), the
// amplitude, and the Gaussian's index within its tile; padded to a multiple of 16 bytes.
//
// Two ways to get y = u (x - b):
//   shifted:  y = u x + nd        D(D+1)/2 FMAs, but the partial sums are as large as |u b|, so the absolute
//             rounding error of y grows with the distance of the Gaussian from the origin in units of its width;
//   centred:  t = x - b, y = u t  D more instructions, error relative to |y| only.
// A Gaussian takes the shifted form iff its `bound` is at most ShiftedBound<T>::v (absolute error of y about
// 2 * unit roundoff * bound: 2e-6 in float, 6e-14 in double).
template <typename T> struct ShiftedBound;
template <> struct ShiftedBound<float> { static constexpr double v = 16.0; };
template <> struct ShiftedBound<double> { static constexpr double v = 256.0; };

template <typename T, int D> struct Rec {
    static constexpr int kU = D * (D + 1) / 2;
    static constexpr int kAmp = kU + D;
    static constexpr int kIdx = kU + D + 1;
    static constexpr int kUsed = kU + D + 1;                                     // 6 / 10 (without the index)
    static constexpr int kStride = (D == 2) ? 8 : 12;
};

template <typename T, int D>
__device__ __forceinline__ void store_record(T* rec, const Derived<D>& d, bool centred, double amplitude, int index) {
    constexpr int kU = Rec<T, D>::kU;
#pragma unroll
    for (int i = 0; i < kU; ++i) rec[i] = T(d.u[i]);
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const double near = d.nd[i], centre = d.b[i];        // (values: a choice between the elements would put d into memory)
        rec[kU + i] = T(centred ? centre : near);
    }
    rec[Rec<T, D>::kAmp] = T(amplitude);
    reinterpret_cast<int*>(rec + Rec<T, D>::kIdx)[0] = index;
}

template <typename T, int D>
__device__ __forceinline__ int record_index(const T* rec) {
    return reinterpret_cast<const int*>(rec + Rec<T, D>::kIdx)[0];
}

// y = u (x - b) in the shifted (CENTRED == false) or centred form; returns q = |y|^2
template <typename T, int D, bool CENTRED>
__device__ __forceinline__ T quad_form(const T* __restrict__ r, const T* __restrict__ x, T* __restrict__ y) {
    if constexpr (D == 2) {
        if constexpr (CENTRED) {
            const T t0 = x[0] - r[3], t1 = x[1] - r[4];
            y[1] = r[2] * t1;
            y[0] = fma_(r[0], t0, r[1] * t1);
        } else {
            y[1] = fma_(r[2], x[1], r[4]);
            y[0] = fma_(r[0], x[0], fma_(r[1], x[1], r[3]));
        }
        return fma_(y[1], y[1], y[0] * y[0]);
    } else {
        if constexpr (CENTRED) {
            const T t0 = x[0] - r[6], t1 = x[1] - r[7], t2 = x[2] - r[8];
            y[2] = r[5] * t2;
            y[1] = fma_(r[3], t1, r[4] * t2);
            y[0] = fma_(r[0], t0, fma_(r[1], t1, r[2] * t2));
        } else {
            y[2] = fma_(r[5], x[2], r[8]);
            y[1] = fma_(r[3], x[1], fma_(r[4], x[2], r[7]));
            y[0] = fma_(r[0], x[0], fma_(r[1], x[1], fma_(r[2], x[2], r[6])));
        }
        return fma_(y[2], y[2], fma_(y[1], y[1], y[0] * y[0]));
    }
}

// acc[p] += amplitude * exp2(-|y|^2) over the records begin, begin + STEP, ... of an LDS tile for the lane's P points.  float:
// the exponentials of all points of a lane at once (pair_exp2_batch), of two Gaussians with three to five points; one and two
// points go one by one.
template <typename T, int D, int P, int STEP, bool CENTRED>
__device__ __forceinline__ void add_pairs(const T* __restrict__ lds, const T* __restrict__ tab, int begin, int end,
                                          const T (&x)[P][D], T (&acc)[P]) {
    constexpr int S = Rec<T, D>::kStride;
    constexpr int U = sizeof(T) == 4 && P >= 3 && P < 6 ? 2 : 1;       // Gaussians whose exponentials are batched
    int g = begin;
    if constexpr (sizeof(T) == 4 && P >= 3) {
        for (; g + (U - 1) * STEP < end; g += U * STEP) {
            T r[U][Rec<T, D>::kUsed], q[U * P], e[U * P];
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int i = 0; i < Rec<T, D>::kUsed; ++i) r[u][i] = lds[(g + u * STEP) * S + i];
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    T y[D];
                    q[u * P + p] = quad_form<T, D, CENTRED>(r[u], x[p], y);
                }
            }
            pair_exp2_batch(q, e);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int p = 0; p < P; ++p) acc[p] = fma_(r[u][Rec<T, D>::kAmp], e[u * P + p], acc[p]);
        }
        if constexpr (U == 1) return;
    }
#pragma unroll 2
    for (; g < end; g += STEP) {
        T r[Rec<T, D>::kUsed];
#pragma unroll
        for (int i = 0; i < Rec<T, D>::kUsed; ++i) r[i] = lds[g * S + i];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            T y[D];
            const T q = quad_form<T, D, CENTRED>(r, x[p], y);
            acc[p] = fma_(r[Rec<T, D>::kAmp], pair_exp2(-q, tab), acc[p]);
        }
    }
}

// Stages up to 256 Gaussians (one per lane of a 256-lane workgroup) into LDS, shifted-form records first,
// centred-form records after them (stable order within each group).  Each of the two groups is padded with null
// records (zero factor and amplitude, index -1) to a multiple of GROUP, so that GROUP consecutive records always
// share one form; the tile needs room for 256 + 2*(GROUP-1) records.  counts[8] receives the start of the
// centred group, counts[9] the padded total.  Contains two workgroup barriers: the first also orders the
// overwrite of the tile after every lane's reads of the previous one, the second publishes the new tile, so the
// caller needs no barrier of its own.
template <typename T, int D, int GROUP = 1>
__device__ __forceinline__ void stage_tile(const T* __restrict__ gaussians, int cnt, double amp_scale, T* lds,
                                           int* counts /* LDS int[10] */, bool covariance_form,
                                           const T* __restrict__ weight_override = nullptr) {
    constexpr int S = Rec<T, D>::kStride;
    constexpr int G = 1 + D + D * D;
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const bool active = tid < cnt;
    Derived<D> dv;
    bool centred = false;
    if (active) {
        dv = derive<T, D>(gaussians + size_t(tid) * G, covariance_form);
        // (the fixed-point fitting evaluates a mixture with other weights than it stores: |x| of the iteration)
        if (weight_override) dv.w = fabs(double(weight_override[tid]));
        centred = !(dv.bound <= ShiftedBound<T>::v);
    }
    const unsigned long long mc = __ballot(active && centred);
    const unsigned long long ms = __ballot(active && !centred);
    if (lane == 0) { counts[wave] = __popcll(ms); counts[4 + wave] = __popcll(mc); }
    __syncthreads();
    int shifted_before = 0, centred_before = 0, shifted_total = 0, centred_total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int cs = counts[w], cc = counts[4 + w];
        if (w < wave) { shifted_before += cs; centred_before += cc; }
        shifted_total += cs;
        centred_total += cc;
    }
    const int centred_start = (shifted_total + GROUP - 1) / GROUP * GROUP;
    const int centred_end = centred_start + centred_total;
    const int padded_total = (centred_end + GROUP - 1) / GROUP * GROUP;
    if (active) {
        const unsigned long long below = (1ull << lane) - 1ull;
        const int slot = centred ? centred_start + centred_before + __popcll(mc & below)
                                 : shifted_before + __popcll(ms & below);
        store_record<T, D>(lds + slot * S, dv, centred, dv.w * dv.norm * amp_scale, tid);
    }
    if constexpr (GROUP > 1) {
        // null records: y = 0, e = 1, amplitude 0 -> no contribution; index -1 -> their sums are dropped
        int slot = -1;
        if (tid < centred_start - shifted_total) slot = shifted_total + tid;
        else if (tid >= GROUP && tid - GROUP < padded_total - centred_end) slot = centred_end + (tid - GROUP);
        if (slot >= 0) {
            T* rec = lds + slot * S;
#pragma unroll
            for (int i = 0; i < Rec<T, D>::kUsed; ++i) rec[i] = T(0);
            reinterpret_cast<int*>(rec + Rec<T, D>::kIdx)[0] = -1;
        }
    }
    if (tid == 0) { counts[8] = centred_start; counts[9] = padded_total; }
    __syncthreads();
}

// Orders the LDS accesses of one wavefront's lanes among themselves (the hardware keeps them in program order).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// stage_tile for ONE wavefront and its own LDS tile: the Gaussian of every lane (already derived; none in lanes with
// active == false) becomes a record, shifted-form ones first, both groups padded with null records to a multiple of
// GROUP.  The index of a record is the lane its Gaussian belongs to.  No workgroup barriers; the tile needs room for
// 64 + 2 (GROUP - 1) records.
struct WaveTile { int centred_start, padded_total; };

template <typename T, int D, int GROUP>
__device__ __forceinline__ WaveTile stage_wave_tile(const Derived<D>& dv, bool active, double amp_scale, T* lds, int lane) {
    constexpr int S = Rec<T, D>::kStride;
    const bool centred = active && !(dv.bound <= ShiftedBound<T>::v);
    const unsigned long long mc = __ballot(centred), ms = __ballot(active && !centred);
    const int shifted_total = __popcll(ms);
    WaveTile t;
    t.centred_start = (shifted_total + GROUP - 1) / GROUP * GROUP;
    const int centred_end = t.centred_start + __popcll(mc);
    t.padded_total = (centred_end + GROUP - 1) / GROUP * GROUP;
    wave_fence();                                            // the tile's previous records have been read
    if (active) {
        const unsigned long long below = (1ull << lane) - 1ull;
        const int slot = centred ? t.centred_start + __popcll(mc & below) : __popcll(ms & below);
        store_record<T, D>(lds + slot * S, dv, centred, dv.w * dv.norm * amp_scale, lane);
    }
    if constexpr (GROUP > 1) {
        int slot = -1;
        if (lane < t.centred_start - shifted_total) slot = shifted_total + lane;
        else if (lane >= GROUP && lane - GROUP < t.padded_total - centred_end) slot = centred_end + (lane - GROUP);
        if (slot >= 0) {
            T* rec = lds + slot * S;
#pragma unroll
            for (int i = 0; i < Rec<T, D>::kUsed; ++i) rec[i] = T(0);
            reinterpret_cast<int*>(rec + Rec<T, D>::kIdx)[0] = -1;
        }
    }
    wave_fence();
    return t;
}

// ---- wavefront (64 lanes) sum; the total arrives in lane 63 -------------------------------------------
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp_mov(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xf, false));
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_mov(double v) {
    // a 64-bit value moves as its two halves; lanes without a source receive 0.0
    const long long bits = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, int(bits), CTRL, ROW_MASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, int(bits >> 32), CTRL, ROW_MASK, 0xf, false);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

template <typename T>
__device__ __forceinline__ T wave_sum_to_lane63(T v) {
    v += dpp_mov<0x111>(v);          // row_shr:1
    v += dpp_mov<0x112>(v);          // row_shr:2
    v += dpp_mov<0x114>(v);          // row_shr:4
    v += dpp_mov<0x118>(v);          // row_shr:8   -> lane 15 of every row holds the row sum
    v += dpp_mov<0x142, 0xa>(v);     // row_bcast:15 into rows 1 and 3
    v += dpp_mov<0x143, 0xc>(v);     // row_bcast:31 into rows 2 and 3 -> lane 63 holds the total
    return v;
}

// ---- sums of 10 or 6 values over the 16 lanes of a DPP row at once ------------------------------------------------
// Lanes 0-7 keep one of two sums and lanes 8-15 the other, then quads and lanes of a quad share out what is left, so
// that one value per lane remains: lane c holds sum row_sums_index<NR>(c).  22 (12) instructions, one LDS store; four
// shifts per pair of sums took 30 (18) and five (three) stores.  The bank masks write only the lanes that keep the sum.
// Written as one block because the compiler has no form for a masked addition whose other lanes stay undefined; a value
// needs two instructions between its write and a DPP read, which the order inside the block and the s_nop in front keep
// (behind it the compiler reads k2 / k1 across lanes, written three instructions before the end).
template <int NR> __device__ __forceinline__ int row_sums_index(int lane) {
    const int b0 = lane & 1, b1 = (lane >> 1) & 1, b2 = (lane >> 2) & 1, b3 = (lane >> 3) & 1;
    if constexpr (NR == 10) return b0 ? (b1 | b2 ? -1 : 8 + b3) : 4 * b1 + 2 * b2 + b3;
    else return b0 | (b1 & b2) ? -1 : b1 ? 4 + b3 : 2 * b2 + b3;
}
__device__ __forceinline__ float row_sums(const float (&s)[10], int lane) {
    float h0, h1, h2, h3, h4, k0, k1, k2;
#define GMC_ROR8(h, a, b) "v_add_f32_dpp " h ", " a ", " a " row_ror:8 row_mask:0xf bank_mask:0x3\n\t" \
                          "v_add_f32_dpp " h ", " b ", " b " row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
#define GMC_MIRROR(k, a, b) "v_add_f32_dpp " k ", " a ", " a " row_half_mirror row_mask:0xf bank_mask:0x5\n\t" \
                            "v_add_f32_dpp " k ", " b ", " b " row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
#define GMC_MIRROR1(k, a) "v_add_f32_dpp " k ", " a ", " a " row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
    asm volatile("s_nop 1\n\t"
                 GMC_ROR8("%[h4]", "%[s8]", "%[s9]") GMC_ROR8("%[h0]", "%[s0]", "%[s1]") GMC_ROR8("%[h1]", "%[s2]", "%[s3]")
                 GMC_ROR8("%[h2]", "%[s4]", "%[s5]") GMC_ROR8("%[h3]", "%[s6]", "%[s7]")
                 GMC_MIRROR1("%[k2]", "%[h4]") GMC_MIRROR("%[k0]", "%[h0]", "%[h1]") GMC_MIRROR("%[k1]", "%[h2]", "%[h3]")
                 : [h0] "=&v"(h0), [h1] "=&v"(h1), [h2] "=&v"(h2), [h3] "=&v"(h3), [h4] "=&v"(h4), [k0] "=&v"(k0),
                   [k1] "=&v"(k1), [k2] "=&v"(k2)
                 : [s0] "v"(s[0]), [s1] "v"(s[1]), [s2] "v"(s[2]), [s3] "v"(s[3]), [s4] "v"(s[4]), [s5] "v"(s[5]),
                   [s6] "v"(s[6]), [s7] "v"(s[7]), [s8] "v"(s[8]), [s9] "v"(s[9]));
    const bool b0 = (lane & 1) != 0, b1 = (lane & 2) != 0;
    const float m0 = (b1 ? k1 : k0) + dpp_mov<0x4e>(b1 ? k0 : k1);       // quad_perm 2 3 0 1
    const float m1 = k2 + dpp_mov<0x4e>(k2);
    return (b0 ? m1 : m0) + dpp_mov<0xb1>(b0 ? m0 : m1);                 // quad_perm 1 0 3 2
}
__device__ __forceinline__ float row_sums(const float (&s)[6], int lane) {
    float h0, h1, h2, k0, k1;
    asm volatile("s_nop 1\n\t"
                 GMC_ROR8("%[h2]", "%[s4]", "%[s5]") GMC_ROR8("%[h0]", "%[s0]", "%[s1]") GMC_ROR8("%[h1]", "%[s2]", "%[s3]")
                 GMC_MIRROR1("%[k1]", "%[h2]") GMC_MIRROR("%[k0]", "%[h0]", "%[h1]")
                 : [h0] "=&v"(h0), [h1] "=&v"(h1), [h2] "=&v"(h2), [k0] "=&v"(k0), [k1] "=&v"(k1)
                 : [s0] "v"(s[0]), [s1] "v"(s[1]), [s2] "v"(s[2]), [s3] "v"(s[3]), [s4] "v"(s[4]), [s5] "v"(s[5]));
    const bool b1 = (lane & 2) != 0;
    const float m = (b1 ? k1 : k0) + dpp_mov<0x4e>(b1 ? k0 : k1);
    return m + dpp_mov<0xb1>(m);
}
#undef GMC_ROR8
#undef GMC_MIRROR
#undef GMC_MIRROR1

// ---- sums over the rows and over the lanes of a row, several values at once ------------------------------------------
// D values of four points per lane, summed over the 16 lanes of a row: afterwards the lanes 4 b ... 4 b + 3 of a row hold
// the sums of point b.  (As in row_sums: masked additions, two instructions between a write and its DPP read.)
__device__ __forceinline__ void row_sums_of_four(const float (&v)[4][3], float (&sum)[3]) {
    float h[6], k[3];
#define GMC_ROR8(h, a, b) "v_add_f32_dpp " h ", " a ", " a " row_ror:8 row_mask:0xf bank_mask:0x3\n\t" \
                          "v_add_f32_dpp " h ", " b ", " b " row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
#define GMC_MIRROR(k, a, b) "v_add_f32_dpp " k ", " a ", " a " row_half_mirror row_mask:0xf bank_mask:0x5\n\t" \
                            "v_add_f32_dpp " k ", " b ", " b " row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
    asm volatile("s_nop 1\n\t"
                 GMC_ROR8("%0", "%9", "%15") GMC_ROR8("%1", "%12", "%18") GMC_ROR8("%2", "%10", "%16")
                 GMC_ROR8("%3", "%13", "%19") GMC_ROR8("%4", "%11", "%17") GMC_ROR8("%5", "%14", "%20")
                 GMC_MIRROR("%6", "%0", "%1") GMC_MIRROR("%7", "%2", "%3") GMC_MIRROR("%8", "%4", "%5") "s_nop 1"
                 : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]), "=&v"(h[4]), "=&v"(h[5]), "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2])
                 : "v"(v[0][0]), "v"(v[0][1]), "v"(v[0][2]), "v"(v[1][0]), "v"(v[1][1]), "v"(v[1][2]),
                   "v"(v[2][0]), "v"(v[2][1]), "v"(v[2][2]), "v"(v[3][0]), "v"(v[3][1]), "v"(v[3][2]));
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        k[d] += dpp_mov<0x4e>(k[d]);                                       // quad_perm 2 3 0 1
        sum[d] = k[d] + dpp_mov<0xb1>(k[d]);                               // quad_perm 1 0 3 2
    }
}
__device__ __forceinline__ void row_sums_of_four(const float (&v)[4][2], float (&sum)[2]) {
    float h[4], k[2];
    asm volatile("s_nop 1\n\t"
                 GMC_ROR8("%0", "%6", "%10") GMC_ROR8("%1", "%8", "%12") GMC_ROR8("%2", "%7", "%11") GMC_ROR8("%3", "%9", "%13")
                 GMC_MIRROR("%4", "%0", "%1") GMC_MIRROR("%5", "%2", "%3") "s_nop 1"
                 : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]), "=&v"(k[0]), "=&v"(k[1])
                 : "v"(v[0][0]), "v"(v[0][1]), "v"(v[1][0]), "v"(v[1][1]), "v"(v[2][0]), "v"(v[2][1]), "v"(v[3][0]), "v"(v[3][1]));
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        k[d] += dpp_mov<0x4e>(k[d]);
        sum[d] = k[d] + dpp_mov<0xb1>(k[d]);
    }
}
#undef GMC_ROR8
#undef GMC_MIRROR
// a and b hold one value per lane each: afterwards the even rows (ROWS = 16) or the lower half (32) hold the sums of a over
// the pairs of rows (halves), the others those of b
template <int ROWS>
__device__ __forceinline__ double swap_sum(double a, double b) {
    const unsigned long long ua = __builtin_bit_cast(unsigned long long, a), ub = __builtin_bit_cast(unsigned long long, b);
    unsigned x[2], y[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const unsigned p = unsigned(ua >> (32 * i)), q = unsigned(ub >> (32 * i));
        if constexpr (ROWS == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(p, q, false, false);
            x[i] = r[0]; y[i] = r[1];
        } else {
            const auto r = __builtin_amdgcn_permlane16_swap(p, q, false, false);
            x[i] = r[0]; y[i] = r[1];
        }
    }
    return __builtin_bit_cast(double, (unsigned long long)(x[1]) << 32 | x[0]) + __builtin_bit_cast(double, (unsigned long long)(y[1]) << 32 | y[0]);
}
// NR = 10 or 6 values per lane summed over the four rows (lanes with the same lane & 15): row r holds the sums
// 4 q + (r >> 1 | (r & 1) << 1) in w[q] for q < NR / 4; the last two sums are in w[NR / 4], the first of them in the rows 0 and 1
// (the same in both), the second in the rows 2 and 3.
template <int NR>
__device__ __forceinline__ void sums_over_rows(const double (&v)[NR], double (&w)[NR / 4 + 1]) {
    static_assert(NR % 4 == 2, "pairs of pairs and one pair");
    double h[NR / 2];
#pragma unroll
    for (int i = 0; i < NR / 2; ++i) h[i] = swap_sum<32>(v[2 * i], v[2 * i + 1]);
#pragma unroll
    for (int q = 0; q < NR / 4; ++q) w[q] = swap_sum<16>(h[2 * q], h[2 * q + 1]);
    w[NR / 4] = swap_sum<16>(h[NR / 2 - 1], h[NR / 2 - 1]);
}

// ---- sum over the 16 lanes of a DPP row; the total arrives in lane 15 of the row ---------------------------
template <typename T>
__device__ __forceinline__ T row_sum_to_lane15(T v) {
    v += dpp_mov<0x111>(v);
    v += dpp_mov<0x112>(v);
    v += dpp_mov<0x114>(v);
    v += dpp_mov<0x118>(v);
    return v;
}

// Sums four values per lane (a, b, c, d) over the 64 lanes at once: the half-wavefronts first exchange the values
// they do not keep (lower half keeps a and c, upper half b and d), then the 16-lane rows of each half do the same,
// and one row reduction is left: the total of a arrives in lane 15, of c in lane 31, of b in lane 47, of d in lane
// 63.  13 vector instructions and 3 cross-lane moves instead of 24 for four separate wavefront sums.
template <typename T>
__device__ __forceinline__ T wave_sum4_to_row_ends(T a, T b, T c, T d, int lane) {
    const bool upper = lane >= 32;
    T keep0 = upper ? b : a, keep1 = upper ? d : c;
    const T send0 = upper ? a : b, send1 = upper ? c : d;
    keep0 += __shfl_xor(send0, 32, 64);
    keep1 += __shfl_xor(send1, 32, 64);
    const bool odd_row = (lane & 16) != 0;
    T keep = odd_row ? keep1 : keep0;
    const T send = odd_row ? keep0 : keep1;
    keep += __shfl_xor(send, 16, 64);
    return row_sum_to_lane15(keep);
}

__device__ __forceinline__ void atomic_add(float* p, float v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void atomic_add(double* p, double v) { unsafeAtomicAdd(p, v); }

template <typename T>
__global__ void fill_zero_kernel(T* p, size_t n) {
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = T(0);
}

// Workgroups are dealt round-robin to the 8 XCDs.  With at least kXcdAffineMin mixtures all point chunks of one
// mixture go to one XCD, so that its L2 serves the repeated reads of the Gaussians (the grid then has
// ceil(n_mixtures / 8) * 8 * chunks workgroups, surplus ones exit); with fewer mixtures chunks are dealt
// plainly, otherwise a single mixture would occupy one XCD only.
constexpr int kXcdAffineMin = 64;

__device__ __forceinline__ void map_workgroup(int id, int chunks, int n_mixtures, int& bl, int& chunk) {
    if (n_mixtures >= kXcdAffineMin) {
        const int xcd = id & 7, slot = id >> 3;
        bl = (slot / chunks) * 8 + xcd;
        chunk = slot % chunks;
    } else {
        bl = id / chunks;
        chunk = id - bl * chunks;
    }
}

inline size_t grid_mixtures(size_t n_mixtures) {
    return n_mixtures >= size_t(kXcdAffineMin) ? (n_mixtures + 7) / 8 * 8 : n_mixtures;
}

// Workgroups of one launch: its threads are counted in 32 bits, and a launch of more starts fewer of them without an error.
inline size_t max_workgroups(int threads) { return ((size_t(1) << 32) - 1) / size_t(threads); }

// A launch with few workgroups (one large mixture, few point chunks) leaves most compute units idle, or with a single
// wavefront per SIMD.  The LDS tiles of Gaussians of a mixture are then dealt to several workgroups per point chunk
// ("slices"), which add their partial results with atomics into outputs that were cleared before.
struct TileSlices { int slices, per_slice; };      // per_slice: Gaussians of a slice (the last one may have fewer)

// Slices of whole LDS tiles, evenly filled: 1280 Gaussians in tiles of 512 are three slices of 432, not 1024 and 256.
// `contended`: the partial results of several mixtures meet on the same addresses, where every slice is one more addition:
// no more slices than asked for, and of whole tiles, so that a short last one ends before the others (dL/dx alone of
// 644 x 2844 Gaussians at 132 shared points, 2-D: twelve even slices 402 us, six 232; 192 x 258 at 27, float64, two even
// ones 29.0, 256 and 2 25.7).
inline TileSlices plan_tile_slices(size_t workgroups, int M, int tile, bool contended = false) {
    const int tiles = (M + tile - 1) / tile;
    TileSlices t{1, M > 0 ? M : 1};
    // sixteen workgroups per compute unit: several scheduling rounds, so that the last one is short (measured on one
    // mixture of 16384 components and 100000 points: 1024 -> 1.80 / 3.96 ms forward / backward in float64, 4096 ->
    // 1.61 / 3.25 ms, no gain beyond; 2.49 / 6.35 ms without slices)
    constexpr size_t kWanted = 4096;
    if (tiles <= 1 || workgroups == 0 || workgroups >= kWanted) return t;
    size_t want = (kWanted + workgroups - 1) / workgroups;
    if (want > size_t(tiles)) want = size_t(tiles);
    if (contended) {
        t.per_slice = (tiles + int(want) - 1) / int(want) * tile;
        t.slices = (M + t.per_slice - 1) / t.per_slice;
        return t;
    }
    const int tiles_per_slice = tiles / int(want);
    const int slices = (tiles + tiles_per_slice - 1) / tiles_per_slice;
    t.per_slice = ((M + slices - 1) / slices + 15) / 16 * 16;
    t.slices = (M + t.per_slice - 1) / t.per_slice;
    return t;
}

// Shader clock under the load of a launch, for benchmark reports.  The clock of the vector ALUs is not a constant
// of the device: with all of them busy it settles well below the peak engine clock, which bounds what a
// compute-bound kernel can reach.  One workgroup in the middle of the grid reads the shader-clock counter and the
// constant-rate counter when it starts and when it ends and leaves the two differences; the counters are scalar
// reads, the values live in scalar registers.
struct ClockProbe {
    long long shader0, wall0;
    bool on;
};
__device__ __forceinline__ ClockProbe clock_probe_begin() {
    ClockProbe c;
    c.on = blockIdx.x == gridDim.x / 2;
    c.shader0 = c.on ? clock64() : 0;
    c.wall0 = c.on ? wall_clock64() : 0;
    return c;
}
__device__ __forceinline__ void clock_probe_end(const ClockProbe& c, long long* __restrict__ out) {
    if (c.on && threadIdx.x == 0) { out[0] = clock64() - c.shader0; out[1] = wall_clock64() - c.wall0; }
}

// Per-Gaussian partial sums of the backward pass, in the transformed coordinates y = u (x - b):
//   R0 = sum_n e g,  R1_i = sum_n e g y_i,  R2_ij = sum_n e g y_i y_j (i <= j)     with e = exp2(-|y|^2)
template <int D> struct Sums { static constexpr int k = 1 + D + D * (D + 1) / 2; };   // 6 / 10

// minimum / maximum over the workgroup of every lane's (lo, hi); thread t < 2D returns component t of
// (min_0..min_D-1, max_0..max_D-1), the other threads return garbage; red[k][0] holds component k for every thread
template <typename T, int D>
__device__ __forceinline__ T block_bounds(const T (&lo)[D], const T (&hi)[D], T (*red)[kBlock]) {
    for (int d = 0; d < D; ++d) { red[d][threadIdx.x] = lo[d]; red[D + d][threadIdx.x] = hi[d]; }
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (int(threadIdx.x) < s)
            for (int d = 0; d < D; ++d) {
                const T a = red[d][threadIdx.x + s], b = red[D + d][threadIdx.x + s];
                if (a < red[d][threadIdx.x]) red[d][threadIdx.x] = a;
                if (b > red[D + d][threadIdx.x]) red[D + d][threadIdx.x] = b;
            }
        __syncthreads();
    }
    return red[threadIdx.x < 2 * D ? threadIdx.x : 0][0];
}

template <typename T>
inline void zero_async(T* p, size_t n, hipStream_t stream) {
    if (n == 0) return;
    const size_t blocks = (n + 255) / 256;
    fill_zero_kernel<T><<<dim3(unsigned(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream>>>(p, n);
}

// two arrays in one launch
template <typename T>
__global__ void fill_zero2_kernel(T* p, size_t n, T* q, size_t m) {
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n + m; i += stride) (i < n ? p[i] : q[i - n]) = T(0);
}
template <typename T>
inline void zero2_async(T* p, size_t n, T* q, size_t m, hipStream_t stream) {
    if (n == 0) return zero_async(q, m, stream);
    if (m == 0) return zero_async(p, n, stream);
    const size_t blocks = (n + m + 255) / 256;
    fill_zero2_kernel<T><<<dim3(unsigned(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream>>>(p, n, q, m);
}

}  // namespace gmc
