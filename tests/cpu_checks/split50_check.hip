// Host check of split50/join50 (pic_device.h) against fix_round128: single
// values up to 2^100 on the grid with ties and both signs, and sums of 2^12
// values kept in the two words.
#include <cmath>
#include <cstdio>
#include <random>

#include "pic_device.h"

using namespace pic;

int main() {
    std::mt19937_64 rng(11);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    long long n = 0, bad = 0;
    auto check = [&](i128 got, i128 want, double at) {
        ++n;
        if (got != want && bad++ < 10) std::printf("at %a\n", at);
    };
    for (int i = 0; i < 3000000; ++i) {
        const int q = (int)(rng() % 200) - 20, k = (int)(rng() % 160) - 60;
        double a = std::ldexp(u(rng), (k > 99 ? 99 : k) - q);
        if (i % 4 == 0) a = std::ldexp(std::floor(std::ldexp(u(rng), 50)) + 0.5, -q);       // ties
        if (i % 4 == 1) a = std::ldexp(std::floor(4 * u(rng)) + u(rng) * 0x1p-40, 50 - q);  // about the words' edge
        u64 lo, hi;
        split50(std::ldexp(a, q), lo, hi);
        check(join50(lo, hi), fix_round128(a, q), a);
    }
    for (int s = 0; s < 200; ++s) {
        const double scale = std::ldexp(1.0, (int)(rng() % 100));
        u64 lo = 0, hi = 0;
        i128 sum = 0;
        for (int i = 0; i < 4096; ++i) {
            const double t = (s & 1 ? std::fabs(u(rng)) : u(rng)) * scale;
            u64 l, h;
            split50(t, l, h);
            lo += l;
            hi += h;
            sum += fix_round128(t, 0);
        }
        check(join50(lo, hi), sum, scale);
    }
    std::printf("%lld values, %lld mismatches\n", n, bad);
    return bad != 0;
}
