// seg16.h -- a particle to a row of 16 lanes, for the small instances whose
// Gaussian stencils would otherwise be a serial chain in one thread: lane e
// holds edge e and weight e of the stencil; and the agent-scope loads and
// stores of values that workgroups exchange inside a launch.
#pragma once
#include "stencil1d.h"
#include "wave_ops.h"

#pragma clang fp contract(off)

namespace pic {

constexpr int kSegLanes = 16;  // lanes per particle

__device__ __forceinline__ u64 ld_agent(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(u64* p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether this block is the last of the launch to arrive (all its threads call;
// everything the others wrote before is visible then).  Clears the ticket.
__device__ __forceinline__ bool last_block(uint32_t* ticket, int32_t* flag) {
    wait_memory();  // every wave's adds have been made before thread 0 announces them
    __syncthreads();
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const uint32_t n = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        *flag = n == gridDim.x - 1 ? 1 : 0;
        if (*flag) {
            __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
    }
    __syncthreads();
    return *flag != 0;
}

// Edge e of the stencil of centre c: f((i - 1/2)/N, c) with i = i0 - R + e
// (src/GaussianFixedPointQuiet.jl:5); lane e of a particle's 16 holds it, and
// weight e = f_{e+1} - f_e comes from the next lane.
template <int R>
__device__ __forceinline__ double seg_weight(double c, double Nd, double iN, int e, int32_t& cell0_, int32_t nmask) {
    const double cN = c * Nd, i0 = rint(cN);
    double f;
    if (edges_fit(cN)) {
        f = gauss_edge<R>(c, i0, e, Nd, iN);
        cell0_ = ((int32_t)(int64_t)i0 - R - 1) & nmask;
    } else {
        f = edge_half_erf((int64_t)i0 - R + e, c, Nd);
        cell0_ = cell0((int64_t)i0 - R, nmask);
    }
    return dpp_f64<0x101>(f, f) - f;  // the next lane's edge (lane 15 has none and no weight)
}

// sum(k -> E[k[1]]*k[2], d(c)): the products on lanes 0..2R, folded left in
// cell order by every lane of the particle (a row of the wave).
template <int R>
__device__ __forceinline__ double seg_fold(double term) {
    double S = dpp_f64<0x150>(term, term);  // row_newbcast: lane q of the row
#define PIC_FOLD(q) S = S + dpp_f64<0x150 + q>(term, term)
    PIC_FOLD(1); PIC_FOLD(2); PIC_FOLD(3); PIC_FOLD(4); PIC_FOLD(5); PIC_FOLD(6); PIC_FOLD(7); PIC_FOLD(8);
    PIC_FOLD(9); PIC_FOLD(10); PIC_FOLD(11); PIC_FOLD(12);
    if constexpr (R == 7) {
        PIC_FOLD(13); PIC_FOLD(14);
    }
#undef PIC_FOLD
    return S;
}

template <int R>
__device__ __forceinline__ double seg_gather(const double* __restrict__ Eld, double c, double Nd, double iN,
                                             int32_t nmask, int e) {
    int32_t first;
    const double wt = seg_weight<R>(c, Nd, iN, e, first, nmask);
    return seg_fold<R>(Eld[(first + e) & nmask] * wt);
}

// r[k[1]] += k[2]*w: lane e <= 2R adds cell i0 - R + e in exact limbs.
template <int R>
__device__ __forceinline__ void seg_deposit(u64* __restrict__ acc, int32_t N, double c, double Nd, double iN,
                                            int32_t nmask, double w, int q, bool fit, int e) {
    int32_t first;
    const double a = seg_weight<R>(c, Nd, iN, e, first, nmask) * w;
    if (e > 2 * R || !(fabs(a) > 0.0)) return;  // NaN adds nothing
    const int32_t cell = (first + e) & nmask;
    if (fit) lds_add_contribution(acc, N, cell, a, q);
    else lds_add_fxp(acc, N, cell, fxp_from(a, q));
}

}  // namespace pic
