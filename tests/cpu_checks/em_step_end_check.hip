// Host check of em_step_end.h: host threads in the place of a block's, with
// thread 0 ahead of all others as far as the barrier lets it.  Every row of
// every step lands in that step's slot, for steps before, in and past the
// slots kept.
#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

#include "em_step_end.h"

using namespace pic;

struct Block {
    std::mutex m;
    std::condition_variable cv;
    int arrived = 0, threads;
    bool first = false;  // thread 0 is at the barrier or past the end
    void go() {
        std::lock_guard<std::mutex> l(m);
        first = true;
        cv.notify_all();
    }
    void wait_first() {
        std::unique_lock<std::mutex> l(m);
        cv.wait(l, [&] { return first; });
    }
    void sync(int t) {
        if (t == 0) go();
        std::unique_lock<std::mutex> l(m);
        ++arrived;
        cv.notify_all();
        cv.wait(l, [&] { return arrived == threads; });
    }
};

static int check(int N, int rows, int threads, int64_t base, int64_t cap, int steps) {
    EM1D s{};
    std::vector<double> out((size_t)(cap * 12 * N), -1.0);
    std::vector<int32_t> sweeps((size_t)cap, -1), ctl(kEMMaxSweeps + 1, 0);
    std::vector<unsigned long long> umax(16, 7);
    int64_t t[2] = {5, base};
    s.N = N;
    s.t = t;
    s.out = out.data();
    s.out_cap = cap;
    s.sweeps_out = sweeps.data();
    s.ctl = ctl.data();
    s.umax = umax.data();
    for (int step = 0; step < steps; ++step) {
        ctl[kEMMaxSweeps] = 100 + step;
        Block b;
        b.threads = threads;
        std::vector<std::thread> ts;
        for (int k = 0; k < threads; ++k)
            ts.emplace_back([&, k] {
                if (k) b.wait_first();
                em_step_end(s, k, threads, rows, [&](int f, int j) { return 1e6 * step + 1000.0 * f + j; },
                            [&] { b.sync(k); });
                if (k == 0) b.go();
            });
        for (std::thread& x : ts) x.join();
    }
    int bad = t[0] != 5 + steps || ctl[0] != 1 || ctl[kEMMaxSweeps] != 0 || umax[1] != 7 || umax[10] != 0;
    for (int64_t slot = 0; slot < cap; ++slot) {
        const int64_t step = slot + base - 5;
        const bool run = step >= 0 && step < steps;
        bad += sweeps[slot] != (run ? 100 + step : -1);
        for (int f = 0; f < 12; ++f)
            for (int j = 0; j < N; ++j)
                bad += out[(slot * 12 + f) * N + j] != (run && f < rows ? 1e6 * step + 1000.0 * f + j : -1.0);
    }
    if (bad) std::printf("N %d rows %d threads %d base %lld cap %lld: %d wrong\n", N, rows, threads, (long long)base,
                         (long long)cap, bad);
    return bad;
}

int main() {
    int bad = 0;
    for (int N : {8, 64, 256})
        for (int rows : {5, 12})
            for (int threads : {1, 3, 16})
                for (int64_t base : {5, 4, 7}) bad += check(N, rows, threads, base, 3, 4);
    std::printf("%d wrong\n", bad);
    return bad != 0;
}
