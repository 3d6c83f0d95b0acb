// wave_ops.h -- lane exchanges inside one 64-lane wave that stay in the vector
// registers (DPP row operations and gfx950's half- and row-swaps), for the
// latency chains of the persistent small-instance kernels.  A __shfl goes
// through the LDS crossbar instead: about 100 cycles of latency a step against
// the 8-16 of these, and a 64-point transform with its convergence test is a
// chain of some 30 of them.
#pragma once
#include "pic_device.h"

#pragma clang fp contract(off)

namespace pic {

// Waits until the wave's stores and atomics have reached the level they are
// performed at.  Before one thread of a block announces the block's work to
// others with an agent-scope release: a block barrier alone does not wait for
// the other waves' outstanding stores.
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// x of the lane that DPP control CTRL names, `old` in the 4-lane banks of a
// row that BANKS leaves out
template <int CTRL, int BANKS = 0xf>
__device__ __forceinline__ double dpp_f64(double old, double x) {
    const u64 o = (u64)__double_as_longlong(old), v = (u64)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)o, (int)(uint32_t)v, CTRL, 0xf, BANKS, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(o >> 32), (int)(v >> 32), CTRL, 0xf, BANKS, false);
    return __longlong_as_double((long long)(((u64)hi << 32) | lo));
}

// the values of lanes l & ~H (lo) and l | H (hi)
template <int H>
__device__ __forceinline__ void lane_pair(double x, double& lo, double& hi) {
    if constexpr (H == 1) {
        lo = dpp_f64<0xA0>(x, x);
        hi = dpp_f64<0xF5>(x, x);
    } else if constexpr (H == 2) {
        lo = dpp_f64<0x44>(x, x);
        hi = dpp_f64<0xEE>(x, x);
    } else if constexpr (H == 4) {
        lo = dpp_f64<0x114, 0xa>(x, x);
        hi = dpp_f64<0x104, 0x5>(x, x);
    } else if constexpr (H == 8) {
        lo = dpp_f64<0x118, 0xc>(x, x);
        hi = dpp_f64<0x108, 0x3>(x, x);
    } else {
        static_assert(H == 16 || H == 32, "a wave has 64 lanes");
        const u64 v = (u64)__double_as_longlong(x);
        const uint32_t a = (uint32_t)v, b = (uint32_t)(v >> 32);
        if constexpr (H == 16) {
            const auto p = __builtin_amdgcn_permlane16_swap(a, a, false, false);
            const auto q = __builtin_amdgcn_permlane16_swap(b, b, false, false);
            lo = __longlong_as_double((long long)(((u64)q[0] << 32) | p[0]));
            hi = __longlong_as_double((long long)(((u64)q[1] << 32) | p[1]));
        } else {
            const auto p = __builtin_amdgcn_permlane32_swap(a, a, false, false);
            const auto q = __builtin_amdgcn_permlane32_swap(b, b, false, false);
            lo = __longlong_as_double((long long)(((u64)q[0] << 32) | p[0]));
            hi = __longlong_as_double((long long)(((u64)q[1] << 32) | p[1]));
        }
    }
}

// The last six steps (h = 32 .. 1) of the canonical tree over the 64 lanes, for
// K values at once; every lane gets the result.  Lane t adds lane t + h as the
// shuffles of tree256 do; lanes past the first half hold the same sums with
// their operands exchanged.  MAX (per value): the NaN-propagating maximum.
template <int K, typename F>
__device__ __forceinline__ void wave_tree(double (&r)[K], F&& op) {
    auto pairs = [&](auto h) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double lo, hi;
            lane_pair<decltype(h)::value>(r[k], lo, hi);
            r[k] = op(k, lo, hi);
        }
    };
    pairs(std::integral_constant<int, 32>{});
    pairs(std::integral_constant<int, 16>{});
    // within a row of 16 a rotation serves: after step h the values repeat
    // every h lanes
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = op(k, r[k], dpp_f64<0x128>(r[k], r[k]));
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = op(k, r[k], dpp_f64<0x124>(r[k], r[k]));
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = op(k, r[k], dpp_f64<0x122>(r[k], r[k]));
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = op(k, r[k], dpp_f64<0x121>(r[k], r[k]));
}

// The sum of v over each group of eight lanes (u64, modulo 2^64), in all of them.
__device__ __forceinline__ u64 sum8_u64(u64 v) {
    auto other = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, C, 0xf, 0xf, false);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(v >> 32), C, 0xf, 0xf, false);
        return ((u64)hi << 32) | lo;
    };
    v += other(std::integral_constant<int, 0xB1>{});   // lane ^ 1
    v += other(std::integral_constant<int, 0x4E>{});   // lane ^ 2
    v += other(std::integral_constant<int, 0x141>{});  // 7 - lane: the other four lanes' sum
    return v;
}

}  // namespace pic
