// em_step_end.h -- the end of a step of the 1D electromagnetic small chain, by
// the threads of one block: the step's output slot (fields[:, t, 1:12]), then
// the step count and the next step's flags.  The slot comes from the count, so
// no thread may move the count before every thread has read it: that is the
// barrier, sync().
#pragma once
#include <hip/hip_runtime.h>

#include "picem1d_internal.h"

namespace pic {

// rows: the fields kept, 12 or, without the moments, 5; value(f, j) is field f
// of cell j (called once for each by the whole block, kept or not)
template <typename Value, typename Sync>
__host__ __device__ __forceinline__ void em_step_end(const EM1D& s, int thread, int threads, int rows, Value&& value,
                                                     Sync&& sync) {
    const int N = s.N;
    const int64_t t = s.t[0], slot = t - s.t[1];
    const int32_t sweeps = s.ctl[kEMMaxSweeps];
    const bool keep = slot >= 0 && slot < s.out_cap;
    double* o = s.out + (keep ? slot : 0) * 12 * N;
    for (int i = thread; i < rows * N; i += threads) {
        const double v = value(i / N, i % N);
        if (keep) o[i] = v;
    }
    sync();
    if (thread != 0) return;
    if (keep) s.sweeps_out[slot] = sweeps;
    s.t[0] = t + 1;
    s.ctl[0] = 1;
    for (int k = 1; k <= kEMMaxSweeps; ++k) s.ctl[k] = 0;
    for (int k = 2; k < kEMMomentMax + 3; ++k) s.umax[k] = 0;
}

}  // namespace pic
