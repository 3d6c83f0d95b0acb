// Host check of gauss_edges.h against the CPU restatement's erf: every interval
// on random arguments and around the branch points, whole stencils (R = 6, 7)
// at random centres, cell edges and cell centres, and the limb split of a
// contribution against fxp_from's definition on 128-bit integers.
//
// With an argument n: the measurement behind tail_delta.  Over n random
// arguments in each of [3, 4], [4, 5] and [5, 6], the largest distance of
// 1 - erfc from the middle of two doubles at which the polynomial's rounding
// differs from the restatement's; fails where it exceeds tail_delta.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#include "gauss_edges.h"

using namespace pic;

extern "C" double orc_erf(double);

static long long n = 0, bad = 0;
static void expect(double got, double want, const char* what, double at) {
    ++n;
    if (__builtin_bit_cast(u64, got) == __builtin_bit_cast(u64, want)) return;
    if (bad++ < 10) std::printf("%s at %a: %a, not %a\n", what, at, got, want);
}

static double inner(int m, double x) {
    d2 c = {0.3, -0.9}, a = {1.1, 1.7}, b = {2.2, 2.9};
    (m == 0 ? c : m == 1 ? a : b)[1] = x;
    erf_inner(c, a, b);
    return (m == 0 ? c : m == 1 ? a : b)[1];
}
static void interval(int m, double x) {
    if (m < 3) {
        expect(inner(m, x), orc_erf(x), "inner", x);
        if (m == 0 && x != 0.0) expect(inner(m, -x), orc_erf(-x), "inner", -x);
        return;
    }
    uint32_t unsure = 0;
    const d2 y = m == 3 ? erf_tail<3>(d2(x), unsure, 0) : m == 4 ? erf_tail<4>(d2(x), unsure, 0)
                                                                  : erf_tail<5>(d2(x), unsure, 0);
    if (!(unsure & 2)) expect(y[1], orc_erf(x), "tail", x);
    if (x < 6.0) expect(erf_tail_full(x), orc_erf(x), "whole form", x);
}

template <int R>
static void stencil(double c, int N) {
    const double Nd = N, i0 = std::rint(c * Nd);
    double f[2 * R + 2];
    gauss_edges<R>(c, i0, Nd, 1.0 / Nd, f);
    for (int j = 0; j < 2 * R + 2; ++j) {
        const long long i = (long long)i0 + j - R;
        const double z = (((double)i - 0.5) / Nd - c) * Nd, e = orc_erf(z) / 2.0;
        // an edge on the centre may carry the other zero
        if (e == 0.0 && f[j] == 0.0) continue;
        expect(f[j], e, "edge", z);
    }
}

template <int M>
static void tail_sweep(long long count, unsigned seed, double* most, long long* differ) {
    std::mt19937_64 rng(seed);
    double far = 0.0;
    long long d = 0;
    for (long long i = 0; i < count; ++i) {
        const double x = M + (double)(rng() >> 11) * 0x1p-53, u = x - (M + 0.5);
        const double a = M == 3 ? erfc_tail3(u) : M == 4 ? erfc_tail4(u) : erfc_tail5(u);
        const double y = 1.0 - a;
        if (y == orc_erf(x)) continue;
        ++d;
        const double at = 0x1p-54 - std::fabs((1.0 - y) - a);
        far = at > far ? at : far;
    }
    *most = far;
    *differ = d;
}
static int tail_sweeps(long long count) {
    const int T = (int)std::max(1u, std::thread::hardware_concurrency());
    int wrong = 0;
    for (int M = 3; M < 6; ++M) {
        std::vector<double> most(T);
        std::vector<long long> differ(T);
        std::vector<std::thread> ts;
        for (int t = 0; t < T; ++t) {
            const long long n = count / T + (t < count % T);
            auto f = M == 3 ? tail_sweep<3> : M == 4 ? tail_sweep<4> : tail_sweep<5>;
            ts.emplace_back(f, n, 100u * M + t, &most[t], &differ[t]);
        }
        double far = 0.0;
        long long d = 0;
        for (int t = 0; t < T; ++t) {
            ts[t].join();
            far = std::max(far, most[t]);
            d += differ[t];
        }
        std::printf("[%d, %d]: %lld arguments, %lld round differently, up to %.2e from the middle (tail_delta %.1e)\n",
                    M, M + 1, count, d, far, tail_delta(M));
        wrong += far > tail_delta(M);
    }
    return wrong;
}

int main(int argc, char** argv) {
    if (argc > 1) return tail_sweeps(std::atoll(argv[1]));
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    for (int i = 0; i < 2000000; ++i)
        for (int m = 0; m < 6; ++m) interval(m, m + u(rng));
    for (int i = 0; i < 200000; ++i) interval(0, std::ldexp(u(rng), -(int)(rng() % 58)));
    interval(0, 0.0);
    const double at[] = {0x1p-60, 0x1p-28, 0.84375, 1.0, 1.25, 2.0, 1 / 0.35, 2.857142, 3.0, 4.0, 5.0, 6.0};
    for (double a : at)
        for (int k = -4; k <= 4; ++k) {
            double x = a;
            for (int s = 0; s < std::abs(k); ++s) x = std::nextafter(x, k < 0 ? -1.0 : 9.0);
            for (int m = 0; m < 6; ++m)
                if (x >= m && x <= m + 1) interval(m, x);
        }
    for (int N = 8; N <= 4096; N *= 2)
        for (int i = 0; i < 4000; ++i) {
            const double k = (double)(rng() % (3 * N)) - N;
            const double cs[] = {u(rng), 3 * u(rng) - 1, k / N, (k + 0.5) / N, std::nextafter((k + 0.5) / N, 9.0),
                                 (k + 0.25) / N, 1e6 * u(rng), 0x1p50 / N * u(rng)};
            for (double c : cs) {
                stencil<6>(c, N);
                stencil<7>(c, N);
            }
        }
    for (int i = 0; i < 2000000; ++i) {
        // values up to 2^126 on the grid; ties included
        double t = std::ldexp(u(rng), (int)(rng() % 170) - 44);
        if (i % 3 == 0) t = std::ldexp(std::floor(std::ldexp(u(rng), 50)) + 0.5, -(int)(i % 2));
        const Limbs43 v = split43(t);
        const u128 got = (u128)small_u64(v.l0) + ((u128)small_u64(v.l1) << 43) + ((u128)small_u64(v.l2) << 86);
        const double r = std::rint(t);
        int e;
        const double f = std::frexp(r, &e);
        const u128 m = (u128)(u64)std::ldexp(f, 53), want = r == 0.0 ? 0 : e >= 53 ? m << (e - 53) : m >> (53 - e);
        ++n;
        if (got != want && bad++ < 10) std::printf("split of %a\n", t);
    }
    std::printf("%lld values, %lld mismatches\n", n, bad);
    return bad != 0;
}
