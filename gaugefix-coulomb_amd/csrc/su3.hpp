// su3.hpp -- register-resident 3x3 complex algebra for the CDNA4 kernels.
//
// All functions are templated on the real type T (float or double) and fully
// unrolled so that every matrix lives in VGPRs (no dynamic register indexing).
// The SU(3) operations restate the reference's group algebra
// (src/SU3_ops.c, src/SU2_ops.c of jesuel-marques/GaugeFix-Coulomb).
#pragma once

#include <hip/hip_runtime.h>

namespace gfc {

template <typename T>
struct alignas(2 * sizeof(T)) cplx {
    T re, im;
};

template <typename T>
struct mat3 {
    cplx<T> e[9];
};

template <typename T>
__device__ __forceinline__ cplx<T> c_make(T re, T im) {
    cplx<T> r;
    r.re = re;
    r.im = im;
    return r;
}

// acc += a * b
template <typename T>
__device__ __forceinline__ void c_mac(cplx<T> &acc, const cplx<T> &a, const cplx<T> &b) {
    acc.re += a.re * b.re;
    acc.re -= a.im * b.im;
    acc.im += a.re * b.im;
    acc.im += a.im * b.re;
}

// acc += a * conj(b)
template <typename T>
__device__ __forceinline__ void c_mac_cb(cplx<T> &acc, const cplx<T> &a, const cplx<T> &b) {
    acc.re += a.re * b.re;
    acc.re += a.im * b.im;
    acc.im += a.im * b.re;
    acc.im -= a.re * b.im;
}

// acc += conj(a) * conj(b)
template <typename T>
__device__ __forceinline__ void c_mac_cc(cplx<T> &acc, const cplx<T> &a, const cplx<T> &b) {
    acc.re += a.re * b.re;
    acc.re -= a.im * b.im;
    acc.im -= a.re * b.im;
    acc.im -= a.im * b.re;
}

// FP64 in explicit FMAs, so that every kernel variant that forms the same
// expression gives the same bits: left to the compiler, the contraction depends
// on the code around it.  (FP32 leaves it to the compiler.)
__device__ __forceinline__ void c_mac(cplx<double> &acc, const cplx<double> &a,
                                      const cplx<double> &b) {
    acc.re = __builtin_fma(-a.im, b.im, __builtin_fma(a.re, b.re, acc.re));
    acc.im = __builtin_fma(a.im, b.re, __builtin_fma(a.re, b.im, acc.im));
}
__device__ __forceinline__ void c_mac_cb(cplx<double> &acc, const cplx<double> &a,
                                         const cplx<double> &b) {
    acc.re = __builtin_fma(a.im, b.im, __builtin_fma(a.re, b.re, acc.re));
    acc.im = __builtin_fma(-a.re, b.im, __builtin_fma(a.im, b.re, acc.im));
}

// a b - c d, and its conjugate
__device__ __forceinline__ cplx<double> c_det2(const cplx<double> &a, const cplx<double> &b,
                                               const cplx<double> &c, const cplx<double> &d) {
    cplx<double> r = c_make<double>(a.re * b.re, a.re * b.im);
    r.re = __builtin_fma(-a.im, b.im, r.re);
    r.re = __builtin_fma(-c.re, d.re, r.re);
    r.re = __builtin_fma(c.im, d.im, r.re);
    r.im = __builtin_fma(a.im, b.re, r.im);
    r.im = __builtin_fma(-c.re, d.im, r.im);
    r.im = __builtin_fma(-c.im, d.re, r.im);
    return r;
}
__device__ __forceinline__ cplx<double> c_conj(const cplx<double> &a) {
    return c_make<double>(a.re, -a.im);
}

// Squared norm of a row.
__device__ __forceinline__ double row_norm(const cplx<double> *r) {
    double n = r[0].re * r[0].re;
    n = __builtin_fma(r[0].im, r[0].im, n);
    n = __builtin_fma(r[1].re, r[1].re, n);
    n = __builtin_fma(r[1].im, r[1].im, n);
    n = __builtin_fma(r[2].re, r[2].re, n);
    return __builtin_fma(r[2].im, r[2].im, n);
}

template <typename T>
__device__ __forceinline__ void m_zero(mat3<T> &m) {
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k] = c_make<T>(0, 0);
}

template <typename T>
__device__ __forceinline__ void m_identity(mat3<T> &m) {
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k] = c_make<T>((k % 4 == 0) ? T(1) : T(0), 0);
}

// c = a * b
template <typename T>
__device__ __forceinline__ void m_mul(const mat3<T> &a, const mat3<T> &b, mat3<T> &c) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cplx<T> s = c_make<T>(0, 0);
#pragma unroll
            for (int k = 0; k < 3; k++) c_mac(s, a.e[3 * i + k], b.e[3 * k + j]);
            c.e[3 * i + j] = s;
        }
}

// acc += a * b^dagger
template <typename T>
__device__ __forceinline__ void m_mac_nd(mat3<T> &acc, const mat3<T> &a, const mat3<T> &b) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int k = 0; k < 3; k++) c_mac_cb(acc.e[3 * i + j], a.e[3 * i + k], b.e[3 * j + k]);
}

template <typename T>
__device__ __forceinline__ mat3<T> m_dagger(const mat3<T> &a) {
    mat3<T> d;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            d.e[3 * i + j] = c_make<T>(a.e[3 * j + i].re, -a.e[3 * j + i].im);
    return d;
}

// acc += a^dagger
template <typename T>
__device__ __forceinline__ void m_add_dagger(mat3<T> &acc, const mat3<T> &a) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            acc.e[3 * i + j].re += a.e[3 * j + i].re;
            acc.e[3 * i + j].im -= a.e[3 * j + i].im;
        }
}

// c = a * b^dagger
template <typename T>
__device__ __forceinline__ void m_mul_nd(const mat3<T> &a, const mat3<T> &b, mat3<T> &c) {
    m_zero(c);
    m_mac_nd(c, a, b);
}

// Third row of an SU(3) matrix from its first two: r2 = conj(r0 x r1).
template <typename T>
__device__ __forceinline__ void m_fill_row2(mat3<T> &m) {
    const cplx<T> *r0 = m.e, *r1 = m.e + 3;
    cplx<T> c0 = c_make<T>(0, 0), c1 = c_make<T>(0, 0), c2 = c_make<T>(0, 0);
    c_mac_cc(c0, r0[1], r1[2]);
    c_mac_cc(c1, r0[2], r1[0]);
    c_mac_cc(c2, r0[0], r1[1]);
    cplx<T> d0 = c_make<T>(0, 0), d1 = c_make<T>(0, 0), d2 = c_make<T>(0, 0);
    c_mac_cc(d0, r0[2], r1[1]);
    c_mac_cc(d1, r0[0], r1[2]);
    c_mac_cc(d2, r0[1], r1[0]);
    m.e[6] = c_make<T>(c0.re - d0.re, c0.im - d0.im);
    m.e[7] = c_make<T>(c1.re - d1.re, c1.im - d1.im);
    m.e[8] = c_make<T>(c2.re - d2.re, c2.im - d2.im);
}

__device__ __forceinline__ void m_fill_row2(mat3<double> &m) {
    const cplx<double> *r0 = m.e, *r1 = m.e + 3;
    m.e[6] = c_conj(c_det2(r0[1], r1[2], r0[2], r1[1]));
    m.e[7] = c_conj(c_det2(r0[2], r1[0], r0[0], r1[2]));
    m.e[8] = c_conj(c_det2(r0[0], r1[1], r0[1], r1[0]));
}

template <typename T>
__device__ __forceinline__ T inv_sqrt(T x);
// FP64: the hardware estimate (v_rsq_f64) and two Newton steps
// y <- y + y (1 - x y^2) / 2, within an ulp or two of 1.0 / sqrt(x) for the
// positive normal x it is used on (norms of the update's SU(2) vectors and
// rows), in a third of the instructions of a square root and a division.
template <>
__device__ __forceinline__ double inv_sqrt<double>(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double t = x * y, e = __builtin_fma(-t, y, 1.0);
    y = __builtin_fma(0.5 * y, e, y);
    t = x * y;
    e = __builtin_fma(-t, y, 1.0);
    return __builtin_fma(0.5 * y, e, y);
}

// 1 / d for d > 0 in FP64: the hardware estimate (v_rcp_f64) and two Newton
// steps y <- y + y (1 - d y), within an ulp of 1.0 / d.
__device__ __forceinline__ double rcp_nr(double d) {
    double y = __builtin_amdgcn_rcp(d);
    double e = __builtin_fma(-d, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-d, y, 1.0);
    return __builtin_fma(y, e, y);
}
template <>
__device__ __forceinline__ float inv_sqrt<float>(float x) {
    return rsqrtf(x);
}

// acc += a b^dagger for SU(3) a and b, where only rows 0 and 1 of a are set:
// rows 0 and 1 of the product from those, row 2 = conj(r0 x r1) (the product
// is in SU(3)): 18 complex products and a 6-product cross product instead of
// 27 and the 6-product rebuild of a's third row.
template <typename T>
__device__ __forceinline__ void m_mac_nd_su3(mat3<T> &acc, const mat3<T> &a, const mat3<T> &b) {
    mat3<T> P;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cplx<T> s = c_make<T>(0, 0);
#pragma unroll
            for (int k = 0; k < 3; k++) c_mac_cb(s, a.e[3 * i + k], b.e[3 * j + k]);
            P.e[3 * i + j] = s;
        }
    m_fill_row2(P);
#pragma unroll
    for (int k = 0; k < 9; k++) acc.e[k] = c_make<T>(acc.e[k].re + P.e[k].re, acc.e[k].im + P.e[k].im);
}

// acc += (a b)^dagger for SU(3) a and b, where only rows 0 and 1 of a are
// set (rows 0 and 1 of a b from those, row 2 by closure).
template <typename T>
__device__ __forceinline__ void m_mac_dagger_su3(mat3<T> &acc, const mat3<T> &a,
                                                 const mat3<T> &b) {
    mat3<T> Q;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cplx<T> s = c_make<T>(0, 0);
#pragma unroll
            for (int k = 0; k < 3; k++) c_mac(s, a.e[3 * i + k], b.e[3 * k + j]);
            Q.e[3 * i + j] = s;
        }
    m_fill_row2(Q);
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            acc.e[3 * i + j] = c_make<T>(acc.e[3 * i + j].re + Q.e[3 * j + i].re,
                                         acc.e[3 * i + j].im - Q.e[3 * j + i].im);
}

// Row r of squared norm n normalised, or left as it is (false) when n is 0.
__device__ __forceinline__ bool scale_row(cplx<double> *r, double n) {
    const bool ok = n != 0.0;
    const double s = inv_sqrt(ok ? n : 1.0);
#pragma unroll
    for (int b = 0; b < 3; b++) r[b] = c_make<double>(r[b].re * s, r[b].im * s);
    return ok;
}

// projectSU3 (src/SU3_ops.c:994-1049): normalise row 0; row 2 = conj(r0 x r1)
// normalised; row 1 = conj(r2 x r0).  Returns false when row 0 or the cross
// product is null; the rows are then written unnormalised, as in the
// reference.
template <typename T>
__device__ __forceinline__ bool m_project_su3(mat3<T> &m) {
    bool ok = true;
    T n0 = 0;
#pragma unroll
    for (int b = 0; b < 3; b++) n0 += m.e[b].re * m.e[b].re + m.e[b].im * m.e[b].im;
    if (n0 != T(0)) {
        T r = inv_sqrt(n0);
#pragma unroll
        for (int b = 0; b < 3; b++) m.e[b] = c_make<T>(m.e[b].re * r, m.e[b].im * r);
    } else {
        ok = false;
    }
    m_fill_row2<T>(m);
    T n2 = 0;
#pragma unroll
    for (int b = 6; b < 9; b++) n2 += m.e[b].re * m.e[b].re + m.e[b].im * m.e[b].im;
    if (n2 != T(0)) {
        T r = inv_sqrt(n2);
#pragma unroll
        for (int b = 6; b < 9; b++) m.e[b] = c_make<T>(m.e[b].re * r, m.e[b].im * r);
    } else {
        ok = false;
    }
    // row 1 = conj(r2 x r0)
    const cplx<T> *r0 = m.e, *r2 = m.e + 6;
    cplx<T> c0 = c_make<T>(0, 0), c1 = c_make<T>(0, 0), c2 = c_make<T>(0, 0);
    c_mac_cc(c0, r2[1], r0[2]);
    c_mac_cc(c1, r2[2], r0[0]);
    c_mac_cc(c2, r2[0], r0[1]);
    cplx<T> d0 = c_make<T>(0, 0), d1 = c_make<T>(0, 0), d2 = c_make<T>(0, 0);
    c_mac_cc(d0, r2[2], r0[1]);
    c_mac_cc(d1, r2[0], r0[2]);
    c_mac_cc(d2, r2[1], r0[0]);
    m.e[3] = c_make<T>(c0.re - d0.re, c0.im - d0.im);
    m.e[4] = c_make<T>(c1.re - d1.re, c1.im - d1.im);
    m.e[5] = c_make<T>(c2.re - d2.re, c2.im - d2.im);
    return ok;
}

__device__ __forceinline__ bool m_project_su3(mat3<double> &m) {
    const bool ok0 = scale_row(m.e, row_norm(m.e));
    m_fill_row2(m);
    const bool ok2 = scale_row(m.e + 6, row_norm(m.e + 6));
    const cplx<double> *r0 = m.e, *r2 = m.e + 6;
    m.e[3] = c_conj(c_det2(r2[1], r0[2], r2[2], r0[1]));
    m.e[4] = c_conj(c_det2(r2[2], r0[0], r2[0], r0[2]));
    m.e[5] = c_conj(c_det2(r2[0], r0[1], r2[1], r0[0]));
    return ok0 && ok2;
}

// Compensated products (two-product and two-sum error terms kept beside the
// sum), for the change of frame at the two ends of a fix: each matrix then
// carries one rounding, as the links of the input do.  FMA contraction is off,
// since the error terms hold for the rounded product.
struct sum2 {
    double hi, lo;
};

__device__ __forceinline__ void s2_mac(sum2 &s, double a, double b) {
#pragma clang fp contract(off)
    const double p = a * b, e = __builtin_fma(a, b, -p);
    const double t = s.hi + p, v = t - s.hi;
    s.lo += e + ((s.hi - (t - v)) + (p - v));
    s.hi = t;
}

// re, im += a * b
__device__ __forceinline__ void s2_cmac(sum2 &re, sum2 &im, const cplx<double> &a,
                                        const cplx<double> &b) {
    s2_mac(re, a.re, b.re);
    s2_mac(re, -a.im, b.im);
    s2_mac(im, a.re, b.im);
    s2_mac(im, a.im, b.re);
}

// Rows [0, R) of hi + lo = (a + alo) b.
template <int R>
__device__ __forceinline__ void m_mul2(const mat3<double> &a, const mat3<double> &alo,
                                       const mat3<double> &b, mat3<double> &hi,
                                       mat3<double> &lo) {
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            sum2 re = {0, 0}, im = {0, 0};
            cplx<double> l = c_make<double>(0, 0);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                s2_cmac(re, im, a.e[3 * i + k], b.e[3 * k + j]);
                c_mac(l, alo.e[3 * i + k], b.e[3 * k + j]);
            }
            hi.e[3 * i + j] = c_make<double>(re.hi, im.hi);
            lo.e[3 * i + j] = c_make<double>(re.lo + l.re, im.lo + l.im);
        }
}

// Row 2 = conj(r0 x r1), each element rounded once.
__device__ __forceinline__ void m_close_row2(mat3<double> &o) {
#pragma unroll
    for (int b = 0; b < 3; b++) {
        const cplx<double> x0 = o.e[(b + 1) % 3], x1 = o.e[3 + (b + 2) % 3];
        const cplx<double> y0 = o.e[(b + 2) % 3], y1 = o.e[3 + (b + 1) % 3];
        sum2 re = {0, 0}, im = {0, 0};
        s2_cmac(re, im, x0, x1);
        s2_cmac(re, im, c_make<double>(-y0.re, -y0.im), y1);
        o.e[6 + b] = c_make<double>(re.hi + re.lo, -(im.hi + im.lo));
    }
}

// The SU(3) matrix nearest hi + lo, whose rows 0 and 1 are orthonormal to
// within some roundings, rounded once: first-order corrections of the rows'
// norms and overlap from compensated sums, row 2 = conj(r0 x r1).  Matrices
// further from SU(3) are projected as elsewhere.
__device__ __forceinline__ void m_polish_su3(const mat3<double> &hi, const mat3<double> &lo,
                                             mat3<double> &m) {
    const cplx<double> *r0 = hi.e, *r1 = hi.e + 3, *l0 = lo.e, *l1 = lo.e + 3;
    sum2 n0 = {-1, 0}, n1 = {-1, 0}, sre = {0, 0}, sim = {0, 0};
    double c0 = 0, c1 = 0;
    cplx<double> cs = c_make<double>(0, 0);
#pragma unroll
    for (int b = 0; b < 3; b++) {
        s2_mac(n0, r0[b].re, r0[b].re);
        s2_mac(n0, r0[b].im, r0[b].im);
        s2_mac(n1, r1[b].re, r1[b].re);
        s2_mac(n1, r1[b].im, r1[b].im);
        s2_cmac(sre, sim, r1[b], c_make<double>(r0[b].re, -r0[b].im));
        c0 += 2 * (r0[b].re * l0[b].re + r0[b].im * l0[b].im);
        c1 += 2 * (r1[b].re * l1[b].re + r1[b].im * l1[b].im);
        c_mac_cb(cs, r1[b], l0[b]);
        c_mac_cb(cs, l1[b], r0[b]);
    }
    const double d0 = -0.5 * (n0.hi + (n0.lo + c0)), d1 = -0.5 * (n1.hi + (n1.lo + c1));
    const cplx<double> s = c_make<double>(-(sre.hi + (sre.lo + cs.re)), -(sim.hi + (sim.lo + cs.im)));
    const double off = 1e-10;
    if (!(fabs(d0) < off && fabs(d1) < off && fabs(s.re) < off && fabs(s.im) < off)) {
        m = hi;
        m_project_su3(m);
        return;
    }
    mat3<double> o;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        cplx<double> k0 = c_make<double>(l0[b].re + d0 * r0[b].re, l0[b].im + d0 * r0[b].im);
        cplx<double> k1 = c_make<double>(l1[b].re + d1 * r1[b].re, l1[b].im + d1 * r1[b].im);
        c_mac(k1, s, r0[b]);
        o.e[b] = c_make<double>(r0[b].re + k0.re, r0[b].im + k0.im);
        o.e[3 + b] = c_make<double>(r1[b].re + k1.re, r1[b].im + k1.im);
    }
    m_close_row2(o);
    m = o;
}

// determinant3x3 (src/SU3_ops.c:251-281), Leibniz expansion along row 0.
template <typename T>
__device__ __forceinline__ cplx<T> m_det(const mat3<T> &m) {
    const cplx<T> *e = m.e;
    cplx<T> c0 = c_make<T>(0, 0), c1 = c_make<T>(0, 0), c2 = c_make<T>(0, 0);
    c_mac(c0, e[4], e[8]);
    c_mac(c1, e[5], e[6]);
    c_mac(c2, e[3], e[7]);
    cplx<T> d0 = c_make<T>(0, 0), d1 = c_make<T>(0, 0), d2 = c_make<T>(0, 0);
    c_mac(d0, e[5], e[7]);
    c_mac(d1, e[3], e[8]);
    c_mac(d2, e[4], e[6]);
    cplx<T> m0 = c_make<T>(c0.re - d0.re, c0.im - d0.im);
    cplx<T> m1 = c_make<T>(c1.re - d1.re, c1.im - d1.im);
    cplx<T> m2 = c_make<T>(c2.re - d2.re, c2.im - d2.im);
    cplx<T> r = c_make<T>(0, 0);
    c_mac(r, e[0], m0);
    c_mac(r, e[1], m1);
    c_mac(r, e[2], m2);
    return r;
}

__device__ __forceinline__ cplx<double> m_det(const mat3<double> &m) {
    const cplx<double> *e = m.e;
    cplx<double> r = c_make<double>(0, 0);
    c_mac(r, e[0], c_det2(e[4], e[8], e[5], e[7]));
    c_mac(r, e[1], c_det2(e[5], e[6], e[3], e[8]));
    c_mac(r, e[2], c_det2(e[3], e[7], e[4], e[6]));
    return r;
}

// The SU(2) element of a Cabibbo-Marinari step on rows (A, B) of w
// (updateSubLosAlamos, src/SU3_ops.c:776-840 with projectSU2,
// src/SU2_ops.c:369-402): x = a/|a| with a = (Re(w_AA + w_BB),
// -Im(w_AB + w_BA), -Re(w_AB - w_BA), -Im(w_AA - w_BB)) maximises
// Re Tr(x w_sub).  For a null a the reference skips the step: false (FP32), or
// x = 1, which leaves the rows as they are (FP64).  A branch around the step
// costs 84 register moves per update with two hits, where its paths join; the
// FP32 sweeps wait for their bytes either way, and straight code would contract
// into other FMAs there and so change their rounding.
template <typename T, int A, int B>
__device__ __forceinline__ bool cm_su2(const mat3<T> &w, T &a0, T &a1, T &a2, T &a3) {
    const cplx<T> waa = w.e[3 * A + A], wbb = w.e[3 * B + B];
    const cplx<T> wab = w.e[3 * A + B], wba = w.e[3 * B + A];
    a0 = waa.re + wbb.re;
    a1 = -(wab.im + wba.im);
    a2 = -(wab.re - wba.re);
    a3 = -(waa.im - wbb.im);
    if constexpr (sizeof(T) == sizeof(double)) {
        const double n = __builtin_fma(a0, a0, __builtin_fma(a1, a1, __builtin_fma(a2, a2, a3 * a3)));
        const bool null = n == 0.0;
        const double r = inv_sqrt(null ? 1.0 : n);
        a0 = null ? 1.0 : a0 * r;
        a1 *= r;
        a2 *= r;
        a3 *= r;
        return true;
    }
    const T s = a0 * a0 + a1 * a1 + a2 * a2 + a3 * a3;
    if (s == T(0)) return false;
    const T r = inv_sqrt(s);
    a0 *= r;
    a1 *= r;
    a2 *= r;
    a3 *= r;
    return true;
}

// Rows A, B of m left-multiplied by the SU(2) element
// [[x0 + i x3, x2 + i x1], [-x2 + i x1, x0 - i x3]].
template <typename T, int A, int B>
__device__ __forceinline__ void cm_rows(mat3<T> &m, T a0, T a1, T a2, T a3) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const cplx<T> p = m.e[3 * A + c], q = m.e[3 * B + c];
        m.e[3 * A + c] = c_make<T>(a0 * p.re - a3 * p.im + a2 * q.re - a1 * q.im,
                                   a0 * p.im + a3 * p.re + a2 * q.im + a1 * q.re);
        m.e[3 * B + c] = c_make<T>(-a2 * p.re - a1 * p.im + a0 * q.re + a3 * q.im,
                                   -a2 * p.im + a1 * p.re + a0 * q.im - a3 * q.re);
    }
}

template <int A, int B>
__device__ __forceinline__ void cm_rows(mat3<double> &m, double a0, double a1, double a2,
                                        double a3) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const cplx<double> p = m.e[3 * A + c], q = m.e[3 * B + c];
        cplx<double> u, v;
        u.re = __builtin_fma(a0, p.re, __builtin_fma(-a3, p.im, __builtin_fma(a2, q.re, -(a1 * q.im))));
        u.im = __builtin_fma(a0, p.im, __builtin_fma(a3, p.re, __builtin_fma(a2, q.im, a1 * q.re)));
        v.re = __builtin_fma(-a2, p.re, __builtin_fma(-a1, p.im, __builtin_fma(a0, q.re, a3 * q.im)));
        v.im = __builtin_fma(-a2, p.im, __builtin_fma(a1, p.re, __builtin_fma(a0, q.im, -(a3 * q.re))));
        m.e[3 * A + c] = u;
        m.e[3 * B + c] = v;
    }
}

template <typename T, int A, int B>
__device__ __forceinline__ void cm_apply(mat3<T> &m, T a0, T a1, T a2, T a3) {
    if constexpr (sizeof(T) == sizeof(double))
        cm_rows<A, B>(m, a0, a1, a2, a3);
    else
        cm_rows<T, A, B>(m, a0, a1, a2, a3);
}

// One Cabibbo-Marinari step on rows (A, B): rows A, B of w and of the
// accumulated update g are left-multiplied by the step's SU(2) element.
template <typename T, int A, int B>
__device__ __forceinline__ void cm_step(mat3<T> &w, mat3<T> &g) {
    T a0, a1, a2, a3;
    if (!cm_su2<T, A, B>(w, a0, a1, a2, a3)) return;
    cm_apply<T, A, B>(w, a0, a1, a2, a3);
    cm_apply<T, A, B>(g, a0, a1, a2, a3);
}

// The first two steps of the first hit, from g = 1 (what cm_step<0, 1> then
// cm_step<0, 2> compute there, without the products with the identity's zeros
// and ones): step (0, 1) sets rows 0, 1 of g to the SU(2) element x, step
// (0, 2) mixes row 0 = (x00, x01, 0) with row 2 = (0, 0, 1).  The values are
// those of the general steps (a product with an exact 0 or 1 is exact).
template <typename T>
__device__ __forceinline__ void cm_first_two(mat3<T> &w, mat3<T> &g) {
    m_identity(g);
    T a0, a1, a2, a3;
    if (cm_su2<T, 0, 1>(w, a0, a1, a2, a3)) {
        cm_apply<T, 0, 1>(w, a0, a1, a2, a3);
        g.e[0] = c_make<T>(a0, a3);
        g.e[1] = c_make<T>(a2, a1);
        g.e[3] = c_make<T>(-a2, a1);
        g.e[4] = c_make<T>(a0, -a3);
    }
    if (!cm_su2<T, 0, 2>(w, a0, a1, a2, a3)) return;
    cm_apply<T, 0, 2>(w, a0, a1, a2, a3);
    // g rows 0 and 2: columns 0, 1 from row 0 alone (row 2 is 0 there),
    // column 2 from row 2 alone (row 0 is 0 there, row 2 is 1)
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const cplx<T> p = g.e[c];
        if constexpr (sizeof(T) == sizeof(double)) {
            g.e[c] = c_make<T>(__builtin_fma(a0, p.re, -(a3 * p.im)),
                               __builtin_fma(a0, p.im, a3 * p.re));
            g.e[6 + c] = c_make<T>(__builtin_fma(-a2, p.re, -(a1 * p.im)),
                                   __builtin_fma(-a2, p.im, a1 * p.re));
        } else {
            g.e[c] = c_make<T>(a0 * p.re - a3 * p.im, a0 * p.im + a3 * p.re);
            g.e[6 + c] = c_make<T>(-a2 * p.re - a1 * p.im, -a2 * p.im + a1 * p.re);
        }
    }
    g.e[2] = c_make<T>(a2, a1);
    g.e[8] = c_make<T>(a0, -a3);
}

// Local Los-Alamos + overrelaxation update from w(n)
// (gaugefixOverrelaxationLocal / updateLosAlamos / power3x3Binomial,
// src/gauge_fixing.c:537-708, src/SU3_ops.c:734-771).
//
// The reference forms g_LA = w_final * w^-1; here the same SU(2) factors are
// accumulated directly into g_LA (g_LA = x_k ... x_1, which equals
// w_final * w^-1 exactly in real arithmetic) -- no complex division and a
// smaller rounding error.  The reference runs the hits only when the real
// part of det(w) is non-zero (inverse3x3 returns the determinant as a double);
// otherwise g_LA = w w^-1 = 1, or g_LA = 0 when det(w) = 0 (the zero inverse).
// Then g_OR = Proj_SU3(1 + omega (g_LA - 1)), or the identity if the
// projection meets a null row.
template <typename T>
__device__ __forceinline__ void la_or_update(mat3<T> &w, int hits, T omega, mat3<T> &g) {
    cplx<T> d = m_det(w);
    if (d.re == T(0)) {
        if (d.im == T(0))
            m_zero(g);
        else
            m_identity(g);
    } else if (hits > 0) {
        cm_first_two(w, g);
        cm_step<T, 1, 2>(w, g);
        for (int h = 1; h < hits - 1; h++) {
            cm_step<T, 0, 1>(w, g);
            cm_step<T, 0, 2>(w, g);
            cm_step<T, 1, 2>(w, g);
        }
        // the last hit outside the loop: the entries of w that no later step
        // reads (row 1's first and row 0's last two columns after (0, 1), rows 0
        // and 2 but for w21, w22 after (0, 2), everything after (1, 2)) are then
        // not computed at all
        if (hits > 1) {
            cm_step<T, 0, 1>(w, g);
            cm_step<T, 0, 2>(w, g);
            cm_step<T, 1, 2>(w, g);
        }
    } else {
        m_identity(g);
    }
#pragma unroll
    for (int k = 0; k < 9; k++) {
        T re = g.e[k].re, im = g.e[k].im;
        if (k % 4 == 0 && sizeof(T) == sizeof(double))
            g.e[k] = c_make<T>(__builtin_fma(omega, re - T(1), T(1)), omega * im);
        else if (k % 4 == 0)
            g.e[k] = c_make<T>(T(1) + omega * (re - T(1)), omega * im);
        else
            g.e[k] = c_make<T>(omega * re, omega * im);
    }
    if (!m_project_su3(g)) m_identity(g);
}

}  // namespace gfc
