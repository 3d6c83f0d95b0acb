// gauss_edges.h -- all edges of a Gaussian stencil at once: erf((g - c)*N) at
// the 2R+2 cell edges around a centre, bit for bit the msun erf of
// pic_device.h (ol_erf), and the cell weights made of them.
//
// What bounds the FP64 Gaussian kernels is the number of FP64 vector
// instructions of these erf.  Called edge by edge in a loop, an erf is a chain
// of branches that a wave walks in full (its lanes' arguments straddle the
// branch points), each division carries the scaling steps of a general
// division, and the edge's argument costs a 64-bit integer conversion and
// another division: about 187 instructions an edge.  Here edge j's argument
// lies in the integer interval [j-R-1, j-R] (the centre is within half a cell
// of its cell), so which branches it can meet is known at compile time:
//   [0, 1]        the two rational forms around 0 and 1, one shared division
//   [1, 2], [2, 3] the exponential form, with one of its neighbours selected
//   [3, 6]        1 - erfc by a polynomial (erfc_tail.h).  It rounds to the
//                 double that msun's 1 - r/x rounds to unless 1 - erfc is
//                 within tail_delta of the middle of two doubles; those (under
//                 1 in 1000) take the exponential form
//   [6, ..)       1
// Centres that are not finite or too far out for exact cell arithmetic take
// the edge-by-edge loop.
//
// Measured on the midpoint push (N = 4096, 3,000,001 particles, a gather and a
// deposit stencil each): 2370 vector instructions per wave in place of 6000,
// 300 us a launch in place of 697, at 72% of the vector issue rate (four waves
// per SIMD: the charge's LDS limbs fill the CU with one block).
//
// The forms and their constants restate FreeBSD msun e_exp.c and s_erf.c, whose
// copyright notices are kept here as their licence asks:
//
// ====================================================
// Copyright (C) 1993 by Sun Microsystems, Inc. All rights reserved.
//
// Developed at SunPro, a Sun Microsystems, Inc. business.
// Permission to use, copy, modify, and distribute this
// software is freely granted, provided that this notice
// is preserved.
// ====================================================
//
// ====================================================
// Copyright (C) 2004 by Sun Microsystems, Inc. All rights reserved.
//
// Permission to use, copy, modify, and distribute this
// software is freely granted, provided that this notice
// is preserved.
// ====================================================
#pragma once
#include "erfc_tail.h"
#include "pic_device.h"

#pragma clang fp contract(off)

#define PIC_HD __host__ __device__ __forceinline__

namespace pic {

// Several edges are evaluated side by side as vectors: a polynomial's constants
// (two scalar moves each) then serve all of them, and their dependent chains
// overlap.  One edge at a time the push of a sweep issued 1140 scalar beside
// 2425 vector instructions per wave.
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));
template <typename T>
struct lanes_of {
    static constexpr int n = sizeof(T) / sizeof(double);
};

PIC_HD uint32_t hi32(double d) { return (uint32_t)(__builtin_bit_cast(u64, d) >> 32); }

// x without its low word.  (By value: a bit cast of a vector's element written
// in place takes its first element.)
PIC_HD double high_part(double x) { return __builtin_bit_cast(double, (u64)hi32(x) << 32); }

// a / b, correctly rounded, for b and a/b well inside the normal range: the
// reciprocal refined twice, then one correction of the quotient -- the steps
// of the compiler's own division without its scaling and special cases, which
// do nothing in that range.
template <typename T>
PIC_HD T div_normal(T a, T b) {
#if defined(__HIP_DEVICE_COMPILE__)
    T r;
    for (int i = 0; i < lanes_of<T>::n; ++i) r[i] = __builtin_amdgcn_rcp(b[i]);
    r = __builtin_elementwise_fma(__builtin_elementwise_fma(-b, r, T(1.0)), r, r);
    r = __builtin_elementwise_fma(__builtin_elementwise_fma(-b, r, T(1.0)), r, r);
    const T q = a * r;
    return __builtin_elementwise_fma(__builtin_elementwise_fma(-b, q, a), r, q);
#else
    return a / b;
#endif
}

// c ? a : b by elements
template <typename T, typename F>
PIC_HD T pick(F&& c, T a, T b) {
    T r;
    for (int i = 0; i < lanes_of<T>::n; ++i) r[i] = c(i) ? a[i] : b[i];
    return r;
}

// msun's erf for |x| in [0.84375, 1.25): erx + P/Q in s = |x| - 1
template <typename T>
PIC_HD void erf_near1(T x, T& P, T& Q) {
    const T s = x - 1.0;
    P = -2.36211856075265944077e-03 +
        s * (4.14856118683748331666e-01 +
             s * (-3.72207876035701323847e-01 +
                  s * (3.18346619901161753674e-01 +
                       s * (-1.10894694282396677476e-01 +
                            s * (3.54783043256182359371e-02 + s * -2.16637559486879084300e-03)))));
    Q = 1.0 +
        s * (1.06420880400844228286e-01 +
             s * (5.40397917702171048937e-01 +
                  s * (7.18286544141962662868e-02 +
                       s * (1.26171219808761642112e-01 +
                            s * (1.36370839120290507362e-02 + s * 1.19844998467991074170e-02)))));
}

// The exponential form's R and S in s = 1/x^2: A below 1/0.35, B from there on
template <typename T>
PIC_HD void erf_RS_A(T s, T& R, T& S) {
    R = -9.86494403484714822705e-03 +
        s * (-6.93858572707181764372e-01 +
             s * (-1.05586262253232909814e+01 +
                  s * (-6.23753324503260060396e+01 +
                       s * (-1.62396669462573470355e+02 +
                            s * (-1.84605092906711035994e+02 +
                                 s * (-8.12874355063065934246e+01 + s * -9.81432934416914548592e+00))))));
    S = 1.0 +
        s * (1.96512716674392571292e+01 +
             s * (1.37657754143519042600e+02 +
                  s * (4.34565877475229228821e+02 +
                       s * (6.45387271733267880336e+02 +
                            s * (4.29008140027567833386e+02 +
                                 s * (1.08635005541779435134e+02 +
                                      s * (6.57024977031928170135e+00 + s * -6.04244152148580987438e-02)))))));
}
template <typename T>
PIC_HD void erf_RS_B(T s, T& R, T& S) {
    R = -9.86494292470009928597e-03 +
        s * (-7.99283237680523006574e-01 +
             s * (-1.77579549177547519889e+01 +
                  s * (-1.60636384855821916062e+02 +
                       s * (-6.37566443368389627722e+02 +
                            s * (-1.02509513161107724954e+03 + s * -4.83519191608651397019e+02)))));
    S = 1.0 +
        s * (3.03380607434824582924e+01 +
             s * (3.25792512996573918826e+02 +
                  s * (1.53672958608443695994e+03 +
                       s * (3.19985821950859553908e+03 +
                            s * (2.55305040643316442583e+03 +
                                 s * (4.74528541206955367215e+02 + s * -2.24409524465858183362e+01))))));
}

// c of msun's exp: x - t*(P1 + t*(P2 + ...)), t = x*x
template <typename T>
PIC_HD T exp_c(T x) {
    const T t = x * x;
    return x - t * (1.66666666666666019037e-01 +
                    t * (-2.77777777770155933842e-03 +
                         t * (6.61375632143793436117e-05 +
                              t * (-1.65339022054652515390e-06 + t * 4.13813679705723846039e-08))));
}

// exp(x) for x in [-40, -1.1]: the argument reduction with k = int(x/ln2 - 1/2)
template <typename T>
PIC_HD T exp_below(T x) {
    T t, pk;
    const T a = 1.44269504088896338700e+00 * x + -0.5;
    for (int i = 0; i < lanes_of<T>::n; ++i) {
        const int32_t k = (int32_t)a[i];
        t[i] = (double)k;
        pk[i] = __builtin_bit_cast(double, (u64)(0x3ff00000u + ((uint32_t)k << 20)) << 32);
    }
    const T hi = x - t * 6.93147180369123816490e-01;
    const T lo = t * 1.90821492927058770002e-10;
    const T r = hi - lo;
    const T c = exp_c(r);
    return (1.0 - ((lo - div_normal(r * c, 2.0 - c)) - hi)) * pk;
}

// exp(x) for |x| in [2^-28, 0.34]: no reduction (k = 0)
template <typename T>
PIC_HD T exp_small(T x) {
    const T c = exp_c(x);
    return 1.0 - (div_normal(x * c, c - 2.0) - x);
}

// exp(-z*z - 0.5625)*exp((z-x)*(z+x) + R/S), z = x without its low word, of
// msun's erf for x in [1, 6): R/S lies in [-0.22, -0.0098] from 1.25 on (above
// -0.34 from 1) and (z-x)(z+x) is below 1.2e-5, so the second exp is
// exp_small's and the first exp_below's
template <typename T>
PIC_HD T erf_exponentials(T x, T R, T S) {
    T z;
    for (int i = 0; i < lanes_of<T>::n; ++i)
        z[i] = high_part(x[i]);
    return exp_below(-z * z - 0.5625) * exp_small((z - x) * (z + x) + div_normal(R, S));
}

// erf(x) for x in [3, 6): the exponential form
PIC_HD double erf_tail_full(double x0) {
    typedef double d1 __attribute__((ext_vector_type(1)));
    const d1 x = d1(x0);
    d1 R, S;
    erf_RS_B(div_normal(d1(1.0), x * x), R, S);
    return (1.0 - div_normal(erf_exponentials(x, R, S), x))[0];
}

// The polynomial's distance from msun's r/x in [M, M+1] is below tail_delta(M):
// in [3, 4] both carry a few roundings of a value below 2.21e-5 (8 units in its
// last place are 4.2e-20), beyond 4 the interpolation error of 1e-21 is the
// larger part.  Over 4e9 random arguments per interval the two rounded
// differently up to 1.02e-20, 8.5e-22 and 9.8e-22 from the middle of two doubles
// (tests/cpu_checks/gauss_edges_check.hip with an argument).
PIC_HD constexpr double tail_delta(int M) { return M == 3 ? 4.2e-20 : 4.0e-21; }

// erf(x) for x in [M, M+1], M = 3, 4, 5; the bits of unsure (from bit `at` on)
// are set where it may not be the rounding of every value within tail_delta(M)
// of 1 - erfc(x)
template <int M>
PIC_HD d2 erf_tail(d2 x, uint32_t& unsure, int at) {
    const d2 u = x - (M + 0.5);
    d2 a;
    if constexpr (M == 3) a = erfc_tail3(u);
    else if constexpr (M == 4) a = erfc_tail4(u);
    else a = erfc_tail5(u);
    const d2 y = 1.0 - a;
    // (1 - y) - a is exact, and at most half of 2^-53, the spacing below 1
    const d2 e = (1.0 - y) - a;
    for (int i = 0; i < 2; ++i)
        if (!(__builtin_fabs(e[i]) <= 0x1p-54 - tail_delta(M)) || (M == 5 && !(x[i] < 6.0))) unsure |= 1u << (at + i);
    return y;
}

// erf of c in [-1, 1], and of a, b in [1, 2] and [2, 3]
PIC_HD void erf_inner(d2& c, d2& a, d2& b) {
    const double erx = 8.45062911510467529297e-01;
    // the form around 1, of |c| and a
    const d4 near = {__builtin_fabs(c[0]), __builtin_fabs(c[1]), a[0], a[1]};
    d4 P, Q;
    erf_near1(near, P, Q);
    // the exponential form of a and b (a below 1.25 has no use for it)
    const d4 x = {a[0], a[1], b[0], b[1]};
    const d4 s = div_normal(d4(1.0), x * x);
    d4 R, S;
    erf_RS_A(s, R, S);
    d2 Rb, Sb;
    erf_RS_B(d2{s[2], s[3]}, Rb, Sb);
    for (int i = 0; i < 2; ++i) {
        const bool far = hi32(b[i]) >= 0x4006DB6Eu;
        R[2 + i] = far ? Rb[i] : R[2 + i];
        S[2 + i] = far ? Sb[i] : S[2 + i];
    }
    const d4 r = erf_exponentials(x, R, S);
    // the form around 0, of c
    const d2 z = c * c;
    const d2 p = 1.28379167095512558561e-01 +
                 z * (-3.25042107247001499370e-01 +
                      z * (-2.84817495755985104766e-02 +
                           z * (-5.77027029648944159157e-03 + z * -2.37630166566501626084e-05)));
    const d2 q = 1.0 + z * (3.97917223959155352819e-01 +
                            z * (6.50222499887672944485e-02 +
                                 z * (5.08130628187576562776e-03 +
                                      z * (1.32494738004321644526e-04 + z * -3.96022827877536812320e-06))));
    d4 n1, n2;
    bool c1[2], a1[2];
    for (int i = 0; i < 2; ++i) {
        c1[i] = hi32(near[i]) >= 0x3feb0000u;
        a1[i] = hi32(a[i]) < 0x3ff40000u;
        n1[i] = c1[i] ? P[i] : p[i];
        n2[i] = c1[i] ? Q[i] : q[i];
        n1[2 + i] = a1[i] ? P[2 + i] : r[i];
        n2[2 + i] = a1[i] ? Q[2 + i] : a[i];
    }
    const d4 y = div_normal(n1, n2);
    const d2 yb = div_normal(d2{r[2], r[3]}, b);
    b = 1.0 - yb;
    for (int i = 0; i < 2; ++i) {
        // |c| < 2^-28: c + efx*c; the edges of a stencil hold no nonzero c below 2^-60
        const double y0 = hi32(near[i]) < 0x3e300000u ? 1.28379167095512586316e-01 : y[i];
        c[i] = c1[i] ? __builtin_copysign(erx + y[i], c[i]) : c[i] + c[i] * y0;
        a[i] = a1[i] ? erx + y[2 + i] : 1.0 - y[2 + i];
    }
}

// erf(z) for |z| in [M, M+1] where M differs from lane to lane: every lane
// evaluates every form and selects its own.
PIC_HD double erf_any(double z, int M) {
    typedef double d1 __attribute__((ext_vector_type(1)));
    const double erx = 8.45062911510467529297e-01;
    const double x = __builtin_fabs(z);
    d1 P, Q, R, S, Rb, Sb;
    erf_near1(d1(x), P, Q);
    const double xe = M >= 1 ? x : 1.5;  // keeps the exponential form's operands in the range of div_normal
    const d1 s = div_normal(d1(1.0), d1(xe * xe));
    erf_RS_A(s, R, S);
    erf_RS_B(s, Rb, Sb);
    const bool far = hi32(xe) >= 0x4006DB6Eu;
    const double r = erf_exponentials(d1(xe), far ? Rb : R, far ? Sb : S)[0];
    const double w = z * z;
    const double p = 1.28379167095512558561e-01 +
                     w * (-3.25042107247001499370e-01 +
                          w * (-2.84817495755985104766e-02 +
                               w * (-5.77027029648944159157e-03 + w * -2.37630166566501626084e-05)));
    const double q = 1.0 + w * (3.97917223959155352819e-01 +
                                w * (6.50222499887672944485e-02 +
                                     w * (5.08130628187576562776e-03 +
                                          w * (1.32494738004321644526e-04 + w * -3.96022827877536812320e-06))));
    const bool near1 = (M == 0 && hi32(x) >= 0x3feb0000u) || (M == 1 && hi32(x) < 0x3ff40000u);
    const bool center = M == 0 && !near1;
    const double y = div_normal(d1(near1 ? P[0] : center ? p : r), d1(near1 ? Q[0] : center ? q : xe))[0];
    if (center) return z + z * (hi32(x) < 0x3e300000u ? 1.28379167095512586316e-01 : y);
    const double e = near1 ? erx + y : hi32(x) >= 0x40180000u ? 1.0 : 1.0 - y;
    return __builtin_copysign(e, z);
}

// f[j] = erf(z_j)/2 for z_j = ((i0 + (j - R - 1/2))/N - c)*N, j = 0..2R+1,
// where i0 = rint(c*N) and |c*N| < 2^51: the edge arguments of the scripts
// (src/GaussianFixedPointQuiet.jl:5), whose (i - 1/2) and, N being a power of
// two, /N are exact.  iN = 1/N.
template <int R>
PIC_HD void gauss_edges(double c, double i0, double Nd, double iN, double (&f)[2 * R + 2]) {
    auto arg = [&](int j) { return ((i0 + ((double)(j - R) - 0.5)) * iN - c) * Nd; };
    // the intervals [M, M+1] on either side: edges R-M (argument < 0) and R+1+M
    auto pair = [&](int M) { return d2{-arg(R - M), arg(R + 1 + M)}; };
    auto put = [&](int M, d2 e) {
        f[R - M] = e[0] * -0.5;
        f[R + 1 + M] = e[1] * 0.5;
    };
#pragma unroll
    for (int M = 6; M <= R; ++M) put(M, d2(1.0));
    d2 e0 = {arg(R), arg(R + 1)}, e1 = pair(1), e2 = pair(2);
    erf_inner(e0, e1, e2);
    f[R] = e0[0] * 0.5;
    f[R + 1] = e0[1] * 0.5;
    put(1, e1);
    put(2, e2);
    uint32_t unsure = 0;
    put(3, erf_tail<3>(pair(3), unsure, 0));
    put(4, erf_tail<4>(pair(4), unsure, 2));
    put(5, erf_tail<5>(pair(5), unsure, 4));
    while (unsure) {  // rare: one copy of the whole form serves the six tails in turn
        const int b = __builtin_ctz(unsure);
        unsure &= unsure - 1;
        const int j = (b & 1) ? R + 4 + (b >> 1) : R - 3 - (b >> 1);
        const double z = __builtin_fabs(arg(j));
        const double e = z < 6.0 ? erf_tail_full(z) * 0.5 : 0.5;
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            if (j == R - 3 - t) f[R - 3 - t] = -e;
            if (j == R + 4 + t) f[R + 4 + t] = e;
        }
    }
}

// One edge of those, j in [0, 2R+1] (lanes of one particle hold one edge each;
// any other j gives a value of no use).
template <int R>
PIC_HD double gauss_edge(double c, double i0, int j, double Nd, double iN) {
    const double z = ((i0 + ((double)(j - R) - 0.5)) * iN - c) * Nd;
    return erf_any(z, j <= R ? R - j : j - R - 1) * 0.5;
}

// A contribution |a| on the 2^-q grid as the three 43-bit limbs of
// lds_add_fxp, in doubles: l0 + l1 2^43 + l2 2^86 = rint(|a| 2^q), ties to even
// (l0 may reach 2^43; every split is exact, so the tie rule of the last one is
// the whole value's).  Valid for |a| 2^q < 2^126.
struct Limbs43 {
    double l0, l1, l2;
};
PIC_HD Limbs43 split43(double t) {  // t = |a| 2^q
    Limbs43 v;
    v.l2 = __builtin_floor(t * 0x1p-86);
    const double r = __builtin_fma(v.l2, -0x1p86, t);
    v.l1 = __builtin_floor(r * 0x1p-43);
    v.l0 = __builtin_rint(__builtin_fma(v.l1, -0x1p43, r));
    return v;
}
// an integer-valued double in [0, 2^52) as u64
PIC_HD u64 small_u64(double v) { return __builtin_bit_cast(u64, v + 0x1p52) & 0xFFFFFFFFFFFFFull; }

}  // namespace pic
