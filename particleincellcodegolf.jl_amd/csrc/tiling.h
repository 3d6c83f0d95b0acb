// tiling.h -- the default tiling of the 1D push launches: every tile of every
// instance holds at most tileP particles and is run by a workgroup of `block`
// threads.  Results do not depend on it.
#pragma once
#include <algorithm>
#include <cstdint>

namespace pic {

struct Tiling {
    int64_t tileP;
    int block;
};

// Members i = 0 .. n - 1 have cells(i) cells and particles(i) particles; fp64:
// the precision; simpson: the Simpson scheme; gauss: a Gaussian stencil; fit:
// workgroups whose LDS fits a CU at once (1 .. 4).
template <typename Cells, typename Particles>
Tiling choose_tiling(int n, Cells&& cells, Particles&& particles, bool fp64, bool simpson, bool gauss, int fit,
                     int numCU) {
    int64_t total = 0;
    double weighted = 0.0;  // sum of a particle's cells
    for (int i = 0; i < n; ++i) {
        total += particles(i);
        weighted += (double)cells(i) * (double)particles(i);
    }
    auto per_tile = [&](int64_t tiles_per_cu) {
        const int64_t target = (int64_t)numCU * tiles_per_cu;
        return (total + target - 1) / target;
    };
    // FP64: as many tiles as fit at once (LDS-bound).  Mixed: two 1024-thread
    // blocks per CU; a single instance below 8192 particles a block takes one
    // (a block's fixed work -- its grid staged, cleared and flushed -- is then
    // half the launch: 83.6 against 93.8 us a step at N = 1024, 3e5 particles;
    // 158.8 against 163.1 at N = 4096, 3e6; two beyond: 353 against 365 us at
    // 2^24).  The Simpson push has more work a particle: below 4096 (N = 64, 2e6
    // particles: 238 against 239.5 us, 2.3e6: 260 against 253, 3.7e6: 339 against
    // 327).
    const int per_cu = fp64 ? fit : (n == 1 && per_tile(2) < (simpson ? 4096 : 8192) ? 1 : 2);
    const Tiling whole = {per_tile(per_cu), fp64 && fit >= 2 ? 512 : 1024};
    if (n == 1 || !gauss) return whole;
    // A batch whose members divide evenly runs all its tiles at once, and
    // smaller ones only add fixed work (mixed, 8 members of 2^20 particles on
    // 4096 cells: 229 us a step, 385 with tiles of 2048; FP64, 8 of 4e5: 998 and
    // 2007 with 1536).  One whose members leave partial tiles has more than fit:
    // the last of them would run alone.  It takes up to 16 smaller tiles per CU,
    // which also spreads out the sweeps that only some members still need, down
    // to 1536 particles or two of a particle's own grids, whose fixed work is
    // then as much as theirs (mixed, 192 members of 32 .. 1024 cells, 9.3e6
    // particles: 286 us a step with 2304-particle tiles, 373 with 18240; 64 such
    // members with the Simpson scheme: 331 with 1536, 354 with 6656).  A few tiles
    // too many are no reason (517 for 512 places, 40 members: 124 us, and 126.5
    // with 1536; 520, 20 of 1e5 particles on 1024 cells: 114, and 101 with 2048).
    const int64_t whole64 = std::max<int64_t>(64, (whole.tileP + 63) / 64 * 64);
    int64_t tiles = 0;
    for (int i = 0; i < n; ++i) tiles += (particles(i) + whole64 - 1) / whole64;
    const int64_t places = (int64_t)numCU * per_cu;
    if (tiles < places + places / 64) return whole;
    const int64_t grids = (int64_t)(2.0 * weighted / (double)total);
    const int64_t small = std::max({per_tile(16), std::min<int64_t>(1536, per_tile(2)), grids});
    if (small >= whole.tileP) return whole;
    return {small, fp64 && fit == 1 ? 1024 : 512};
}

}  // namespace pic
