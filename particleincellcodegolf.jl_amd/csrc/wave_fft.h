// wave_fft.h -- transforms of up to 512 points and the canonical norms inside one
// wave, for the kernels whose small grids make them a latency chain: the lane
// exchanges stay in registers (wave_ops.h), and so do a lane's twiddles.
//
// Element i of an N-point transform lives in lane i % 64, slot i / 64 < E (E = 1
// up to N = 64).  A radix-2 stage with half-size h < 64 pairs lanes l and l ^ h,
// with h >= 64 slots q and q + h/64 of one lane; every butterfly is the
// stage-by-stage transform's (operands b = the upper element, a = the lower,
// t = b w, a + t and a - t; twiddle of stage s at table entry 2^(s-1) - 1 + j,
// conjugated for the inverse), so the result is that of the CPU restatement bit
// for bit.
#pragma once
#include "wave_ops.h"

#pragma clang fp contract(off)

namespace pic {

// A lane's twiddles of the stages with h < 64.
__device__ __forceinline__ void load_wave_twiddles(double2 (&w6)[6], const double2* __restrict__ tw, int N) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        const int h = 1 << s;
        w6[s] = h < N ? tw[h - 1 + (l & (h - 1))] : double2{0.0, 0.0};
    }
}

// x with its sign flipped where `upper`
__device__ __forceinline__ double flip_if(bool upper, double x) {
    return __longlong_as_double(__double_as_longlong(x) ^ (upper ? (long long)0x8000000000000000ull : 0ll));
}

template <int E, int H>
__device__ __forceinline__ void wave_stage(double (&re)[E], double (&im)[E], double wr, double wi) {
    const bool upper = (threadIdx.x & H) != 0;
#pragma unroll
    for (int q = 0; q < E; ++q) {
        double ar, ai, br, bi;
        lane_pair<H>(re[q], ar, br);
        lane_pair<H>(im[q], ai, bi);
        const double tr = br * wr - bi * wi;
        const double tq = br * wi + bi * wr;
        re[q] = ar + flip_if(upper, tr);  // a - t is a + (-t)
        im[q] = ai + flip_if(upper, tq);
    }
}

template <int E>
__device__ __forceinline__ void wave_radix2(double (&re)[E], double (&im)[E], const double2 (&w6)[6],
                                            const double2* __restrict__ tw, int N, bool inverse) {
    auto wi = [&](int s) { return inverse ? -w6[s].y : w6[s].y; };
    if (N > 1) wave_stage<E, 1>(re, im, w6[0].x, wi(0));
    if (N > 2) wave_stage<E, 2>(re, im, w6[1].x, wi(1));
    if (N > 4) wave_stage<E, 4>(re, im, w6[2].x, wi(2));
    if (N > 8) wave_stage<E, 8>(re, im, w6[3].x, wi(3));
    if (N > 16) wave_stage<E, 16>(re, im, w6[4].x, wi(4));
    if (N > 32) wave_stage<E, 32>(re, im, w6[5].x, wi(5));
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int hs = 1; hs < E; hs <<= 1) {
        const int h = hs * 64;
#pragma unroll
        for (int q = 0; q < E; ++q) {
            if (q & hs) continue;
            const double2 w = tw[h - 1 + ((q * 64 + l) & (h - 1))];
            const double wr = w.x, wq = inverse ? -w.y : w.y;
            const double br = re[q + hs], bi = im[q + hs];
            const double tr = br * wr - bi * wq;
            const double tq = br * wq + bi * wr;
            const double ar = re[q], ai = im[q];
            re[q] = ar + tr;
            im[q] = ai + tq;
            re[q + hs] = ar - tr;
            im[q + hs] = ai - tq;
        }
    }
}

// The canonical reduction tree (tree256 over lanes t < 256 that each fold the
// elements t, t + 256, ... from +0.0) of K arrays of N <= 512 values in one wave:
// tree lane t = l + 64u folds slots u, u + 4 of lane l, the two halving steps combine
// (u, u + 2) and then (0, 1) in lane l, and the last six steps are wave_tree's.
// op(k, a, b): array k's sum or NaN-propagating maximum.  Every value is >= 0
// (squares, magnitudes, flags), so folding +0.0 for a missing element leaves a
// sum or maximum unchanged.
template <int K, int E, typename F>
__device__ __forceinline__ void wave_canon(double (&r)[K], const double (&x)[K][E], F&& op) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double P[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            P[u] = 0.0;
#pragma unroll
            for (int q = u; q < E; q += 4) P[u] = op(k, P[u], x[k][q]);
        }
        r[k] = E > 2 ? op(k, op(k, P[0], P[2]), op(k, P[1], P[3])) : E > 1 ? op(k, P[0], P[1]) : P[0];
    }
    wave_tree<K>(r, op);
}

// In one wave: block_isapprox's norms and decisions for isapprox(F, E) on N
// values (lane l, slot q holds element 64 q + l; 0 past N); max |E| and the
// canonical sum of E^2 beside it.
template <int E>
__device__ __forceinline__ bool wave_isapprox(const double (&f)[E], const double (&e)[E], int N, double rtol, double& me,
                                              double& se) {
    const int l = threadIdx.x & 63;
    bool conv;
    // the three norms of block_norms3: d = F - E, F, E; maxima 0..2, sums of squares 3..5
    double x[6][E], r[6];
    auto op = [](int k, double a, double b) { return k < 3 ? nanmax(a, b) : a + b; };
    auto val = [&](int v, int q) { return v == 0 ? f[q] - e[q] : (v == 1 ? f[q] : e[q]); };
#pragma unroll
    for (int v = 0; v < 3; ++v)
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const double xv = val(v, q);
            x[v][q] = fabs(xv);
            x[3 + v][q] = xv * xv;
        }
    wave_canon<6, E>(r, x, op);
    me = r[2];
    se = r[5];
    double nrm[3];
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        const double m = r[v];
        const bool direct = m == 0.0 || isinf(m);
        const bool scaled = !direct && !(isfinite((double)N * m * m) && m * m != 0.0);
        double s = r[3 + v];
        if (scaled) {
            double y[1][E], t[1];
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const double z = q * 64 + l < N ? fabs(val(v, q)) / m : 0.0;
                y[0][q] = z * z;
            }
            wave_canon<1, E>(t, y, [](int, double a, double b) { return a + b; });
            s = t[0];
        }
        nrm[v] = direct ? m : (scaled ? m * sqrt(s) : sqrt(s));
    }
    const double dn = nrm[0], nf = nrm[1], ne = nrm[2];
    if (isfinite(dn)) {
        double mx = nf > ne ? nf : ne;
        if (nf != nf || ne != ne) mx = __longlong_as_double(0x7ff8000000000000LL);
        const double tol = rtol * mx;
        double lim = 0.0 > tol ? 0.0 : tol;
        if (tol != tol) lim = tol;
        conv = dn <= lim;
    } else {
        double y[1][E], t[1];
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const double a = f[q], b = e[q];
            bool good = a == b;
            if (!good && isfinite(a) && isfinite(b)) {
                const double ma = fabs(a) > fabs(b) ? fabs(a) : fabs(b);
                const double tl = rtol * ma;
                good = fabs(a - b) <= (0.0 > tl ? 0.0 : tl);
            }
            y[0][q] = good ? 0.0 : 1.0;
        }
        wave_canon<1, E>(t, y, [](int, double a, double b) { return nanmax(a, b); });
        conv = t[0] == 0.0;
    }
    return conv;
}

}  // namespace pic
