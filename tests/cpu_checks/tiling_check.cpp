// Prints the default tiling (csrc/tiling.h) of a batch: argv = fp64 simpson
// gauss fit numCU, then the members' cells and particles.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "tiling.h"

int main(int argc, char** argv) {
    std::vector<long> a;
    for (int i = 1; i < argc; ++i) a.push_back(std::atol(argv[i]));
    const pic::Tiling t = pic::choose_tiling(
        (argc - 6) / 2, [&](int i) { return a[5 + 2 * i]; }, [&](int i) { return a[6 + 2 * i]; }, a[0] != 0, a[1] != 0,
        a[2] != 0, (int)a[3], (int)a[4]);
    std::printf("%lld %d\n", (long long)t.tileP, t.block);
}
