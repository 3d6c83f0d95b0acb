// kernels_small.hip -- persistent FP64 kernels for small single instances: the
// whole step loop of a run (src/NGPFourier.jl:4-7, src/Gaussian.jl:8-11,
// src/GaussianFixedPointQuiet.jl:7-13) in one launch, with the Picard sweeps
// and their convergence test on the device and no host round trip or graph
// node between steps.
//
// At N <= 256 and a few thousand particles a step is a chain of tiny
// dependent phases (deposit, solve, test, gather) whose cost in the captured
// graph is launch latency, not work.  Two kernels remove it:
//
//  k_small_ngp    one workgroup of 512 threads; the particles stay in
//                 registers for the whole run (thread t owns particles
//                 t + 512 j), counts per cell in LDS, the solve in LDS.
//  k_small_gauss  the Gaussian stencils, whose 16 erf per centre are too much
//                 arithmetic for one compute unit: K particle workgroups with
//                 16 lanes per particle (lane e evaluates edge e of the
//                 stencil, so one wave carries 4 particles and a stencil costs
//                 one erf of latency), plus one diagnostics workgroup.  Each
//                 Picard iteration deposits into LDS limbs, adds them to a
//                 device accumulator, meets at one grid barrier, and then
//                 every workgroup solves the field redundantly (N <= 256 is a
//                 few microseconds in one wave), runs the same convergence test on
//                 the same bits and gathers.  The launch is cooperative, so
//                 all workgroups are resident; every barrier wait is bounded.
//
// Both produce the same bits as the graph path (and the CPU restatement):
// the same stencil expressions, exact integer charge sums, the same solve and
// the same reduction trees.  Compiled with -ffp-contract=off.
#include "pic_device.h"
#include "pic_internal.h"
#include "seg16.h"
#include "solve1d.h"
#include "stencil1d.h"
#include "wave_fft.h"

#pragma clang fp contract(off)

namespace pic {

constexpr int kSmallThreads = kSolveThreads;  // threads per workgroup of both kernels
constexpr int kSegs = kSmallThreads / kSegLanes;

// LDS layout shared by both kernels (doubles): the charge (bit-reversed), the
// solve's permutation (re, im), the previous field, the field, reduction
// scratch, diagnostics partials, the solve's tables (stage twiddles of an
// N-point transform as double2, then the 1/(2 pi k) factors) and the u64
// charge counters (NGP: N counts; Gaussian: 3 N limbs).
__host__ __device__ constexpr int small_lds_doubles(int N) {
    return 5 * N + kRedDoubles + 8 + 2 * N + (N / 2 + 1) + 3 * N;
}
int small_lds_bytes(int N) { return 8 * small_lds_doubles(N); }

struct SmallLds {
    double *re, *bre, *bim, *Fl, *red, *Eld, *dp, *xi;
    double2* tw;
    u64* acc;
};

__device__ __forceinline__ SmallLds small_lds(double* sm, int N) {
    SmallLds L;
    L.re = sm;
    L.bre = sm + N;
    L.bim = sm + 2 * N;
    L.Fl = sm + 3 * N;
    L.Eld = sm + 4 * N;
    L.red = sm + 5 * N;
    L.dp = L.red + kRedDoubles;
    L.tw = reinterpret_cast<double2*>(L.dp + 8);
    L.xi = L.dp + 8 + 2 * N;
    L.acc = reinterpret_cast<u64*>(L.xi + N / 2 + 1);
    return L;
}

// Stages the solve's tables in LDS: the stage twiddles an N-point transform
// reads (entries below N - 1) and the factors 1/(2 pi k), k <= N/2.
__device__ __forceinline__ void stage_tables(const SmallLds& L, const double2* __restrict__ tw, int N) {
    const double* xi = reinterpret_cast<const double*>(tw) + kXiOffset;
    for (int i = threadIdx.x; i < N; i += blockDim.x) L.tw[i] = tw[i];
    for (int i = threadIdx.x; i <= N / 2; i += blockDim.x) L.xi[i] = xi[i];
    __syncthreads();
}

// ---------------------------------------------------------------------------
// The solve in one wave (wave_fft.h); its latency chain takes 5300 cycles at
// N = 64 with the test, where lane shuffles through LDS took 12800.
// ---------------------------------------------------------------------------

// What a lane of wave 0 keeps of the tables.
template <int E>
struct WaveTables {
    double2 w[6];  // its twiddle of the stages with h < 64
    double xt[E];  // 1/(2 pi k') of its modes
};

template <int E>
__device__ __forceinline__ void load_wave_tables(WaveTables<E>& W, const SmallLds& L, int N) {
    const int l = threadIdx.x & 63;
    load_wave_twiddles(W.w, L.tw, N);
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int m = q * 64 + l;
        W.xt[q] = m >= N ? 0.0 : m == 0 ? L.xi[1] : (m <= N / 2 ? L.xi[m] : -L.xi[N - m]);
    }
}

// In wave 0: the solve of the charge staged in L.re (bit-reversed),
// E = real(ifft((xi = fft(rho) ./ ik; xi[1] *= 0; xi))) into Eld, with ik and
// Julia's division by (0, 2 pi k') as in k_solve; with TEST also the
// convergence test isapprox(Fl, E) of the midpoint loop, with block_isapprox's
// norms and decisions (Fl then takes E).  red gets max |E|, the test's result
// and the canonical sum of E^2.
template <bool TEST, int E>
__device__ __forceinline__ void wave_solve(const SmallLds& L, const WaveTables<E>& W, int N, int log2N, double rtol) {
    const int l = threadIdx.x;
    double re[E], im[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int i = q * 64 + l;
        re[q] = i < N ? L.re[i] : 0.0;
        im[q] = 0.0;
    }
    double f[E];
    if (TEST)
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int i = q * 64 + l;
            f[q] = i < N ? L.Fl[i] : 0.0;
        }
    wave_radix2<E>(re, im, W.w, L.tw, N, false);
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int m = q * 64 + l;
        if (m >= N) continue;
        double a = im[q] * W.xt[q];
        double b = -(re[q] * W.xt[q]);
        if (m == 0) {
            a = a * 0.0;
            b = b * 0.0;
        }
        const int p = (int)brev((uint32_t)m, log2N);
        L.bre[p] = a;
        L.bim[p] = b;
    }
    // the permutation stays inside the wave: LDS operations of one wave
    // complete in order; the fences keep the compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int i = q * 64 + l;
        re[q] = i < N ? L.bre[i] : 0.0;
        im[q] = i < N ? L.bim[i] : 0.0;
    }
    wave_radix2<E>(re, im, W.w, L.tw, N, true);
    const double scale = 1.0 / (double)N;
    double e[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int i = q * 64 + l;
        e[q] = i < N ? re[q] * scale : 0.0;
        if (i < N) L.Eld[i] = e[q];
    }
    bool conv = false;
    double me, se;
    if (TEST) {
        conv = wave_isapprox<E>(f, e, N, rtol, me, se);
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int i = q * 64 + l;
            if (i < N) L.Fl[i] = e[q];
        }
    } else {
        double x[2][E], r[2];
#pragma unroll
        for (int q = 0; q < E; ++q) {
            x[0][q] = fabs(e[q]);
            x[1][q] = e[q] * e[q];
        }
        wave_canon<2, E>(r, x, [](int k, double a, double b) { return k < 1 ? nanmax(a, b) : a + b; });
        me = r[0];
        se = r[1];
    }
    if (l == 0) {
        L.red[0] = me;
        L.red[1] = conv ? 1.0 : 0.0;
        L.red[2] = se;
    }
}

// D[t,1:4] of one step from the canonical sum of E^2 and the chunk partials in
// dp (src/GaussianFixedPointQuiet.jl:11,13), as k_diag_final writes it: the
// tree over at most four partials is (p0 + p2) + (p1 + p3) with +0.0 for the
// missing ones, each folded from +0.0.  One thread calls it.
__device__ __forceinline__ void small_diag_row(const SmallLds& L, const InstDesc& I, double se, int nch,
                                               double* __restrict__ row4, int32_t* __restrict__ sweeps,
                                               int32_t nsweeps) {
    double p[2][4];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) p[k][c] = c < nch ? 0.0 + L.dp[2 * c + k] : 0.0;
    const double sv = (p[0][0] + p[0][2]) + (p[0][1] + p[0][3]), sp = (p[1][0] + p[1][2]) + (p[1][1] + p[1][3]);
    const double d1 = (se / (double)I.N) / 2.0;
    const double d2 = ((sv * I.W) / (double)I.P) / 2.0;
    const double d3 = d1 + d2;
    const double s = 2.0 / I.W;
    row4[0] = d1 * s;
    row4[1] = d2 * s;
    row4[2] = d3 * s;
    row4[3] = sp;
    *sweeps = nsweeps;
}

// v/P as the reference divides it: by the exact reciprocal where P is a power
// of two
struct DivP {
    double P, rP;
    bool pow2;
    __device__ __forceinline__ explicit DivP(int64_t n) : P((double)n), rP(1.0 / (double)n), pow2((n & (n - 1)) == 0) {}
    __device__ __forceinline__ double operator()(double v) const { return pow2 ? v * rP : v / P; }
};

// ---------------------------------------------------------------------------
// NGP leapfrog (src/NGPFourier.jl:4-6), one workgroup.  Thread t holds lane
// t % 256 of diagnostics chunk t / 256 (particles 4096 (t / 256) + t % 256 +
// 256 i, i < 16), so the sums of a chunk's lanes need no exchange; their trees
// run in waves 1 and 2 beside the next step's solve in wave 0.
// ---------------------------------------------------------------------------
template <int E>
__global__ void __launch_bounds__(kSmallThreads)
k_small_ngp(SmallRun a) {
    extern __shared__ double sm[];
    constexpr int J = kSmallNgpSlots;
    static_assert(J * kTreeLanes == kTreeChunk && kSmallThreads == 2 * kTreeLanes, "one lane of one chunk per thread");
    const InstDesc I = a.I;
    InstState S = *a.st;
    const int N = I.N, log2N = I.log2N;
    const SmallLds L = small_lds(sm, N);
    const int t = threadIdx.x;
    const int64_t P = I.P;
    const double Nd = (double)N, dt = I.dt;
    const DivP divP(P);
    const int32_t nmask = I.nmask;
    const int par0 = S.step & 1;
    const double* X = par0 ? a.X1 : a.X0;
    const double* V = par0 ? a.V1 : a.V0;
    double x[J], v[J];
    bool has[J];
    const int64_t p0 = (int64_t)(t / kTreeLanes) * kTreeChunk + (t % kTreeLanes);
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int64_t p = p0 + (int64_t)kTreeLanes * j;
        has[j] = p < P;
        x[j] = has[j] ? X[p] : 0.0;
        v[j] = has[j] ? V[p] : 0.0;
    }
    stage_tables(L, a.tw, N);
    WaveTables<E> W;
    load_wave_tables<E>(W, L, N);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(L.acc);
    for (int c = t; c < N; c += kSmallThreads) cnt[c] = 0;
    const u128 one = fxp_from(I.w, I.q);
    const int nch = (int)((P + kTreeChunk - 1) / kTreeChunk);
    double se = 0.0;  // of the step whose row is still to be written
    bool bad = false;
    __syncthreads();
    // the trees of chunk c's lane sums (L.red + 16 + 512 k + 256 c) into dp
    auto trees = [&](int c) {
        const int l = t & 63;
        double r[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const double* q = L.red + 16 + 512 * k + kTreeLanes * c + l;
            r[k] = (q[0] + q[128]) + (q[64] + q[192]);
        }
        wave_tree<2>(r, [](int, double x1, double x2) { return x1 + x2; });
        if (l == 0) {
            L.dp[2 * c] = r[0];
            L.dp[2 * c + 1] = r[1];
        }
    };
    for (int64_t s = 0; s < a.nsteps; ++s) {
        // u(); n[f(j)] += w (the count; times w exactly below)
#pragma unroll
        for (int j = 0; j < J; ++j)
            if (has[j]) {
                x[j] = jl_mod1f(x[j] + (v[j] / 2.0) * dt);
                atomicAdd(&cnt[ngp_cell(x[j], Nd, nmask)], 1u);
            }
        __syncthreads();
        for (int c = t; c < N; c += kSmallThreads) {
            L.re[(int)brev((uint32_t)c, log2N)] = fxp_to((u128)cnt[c] * one, I.q);
            cnt[c] = 0;
        }
        __syncthreads();
        if (t < 64) wave_solve<false, E>(L, W, N, log2N, 0.0);
        else if (s > 0 && t < 64 * (1 + nch)) trees((t >> 6) - 1);
        __syncthreads();
        bad = bad || !isfinite(L.red[0]);
        if (s > 0 && t == kSmallThreads - 1) small_diag_row(L, I, se, nch, a.diag + 4 * (s - 1), a.sweeps + s - 1, 1);
        se = L.red[2];
        // u(); v += E[f.(x)]*dt; the lane's sums of v^2 and v/P in order
        double s2 = 0.0, s1 = 0.0;
#pragma unroll
        for (int j = 0; j < J; ++j)
            if (has[j]) {
                x[j] = jl_mod1f(x[j] + (v[j] / 2.0) * dt);
                v[j] = v[j] + L.Eld[ngp_cell(x[j], Nd, nmask)] * dt;
                s2 = s2 + v[j] * v[j];
                s1 = s1 + divP(v[j]);
            }
        L.red[16 + t] = s2;
        L.red[16 + 512 + t] = s1;
    }
    __syncthreads();
    if (a.nsteps > 0 && t < 64 * nch) trees(t >> 6);
    __syncthreads();
    if (a.nsteps > 0 && t == 0) small_diag_row(L, I, se, nch, a.diag + 4 * (a.nsteps - 1), a.sweeps + a.nsteps - 1, 1);
    const int parN = (int)((S.step + a.nsteps) & 1);
    double* Xo = parN ? a.X1 : a.X0;
    double* Vo = parN ? a.V1 : a.V0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int64_t p = p0 + (int64_t)kTreeLanes * j;
        if (has[j]) {
            Xo[p] = x[j];
            Vo[p] = v[j];
        }
    }
    for (int c = t; c < N; c += kSmallThreads) a.E0[c] = L.Eld[c];
    if (t == 0) {
        S.step += (int32_t)a.nsteps;
        S.e_cur = 0;
        S.last_sweep = 0;
        if (bad) S.err |= 1;
        *a.st = S;
    }
}

// ---------------------------------------------------------------------------
// Grid barrier of k_small_gauss.  Each workgroup has a word of its own, which
// takes the generation it arrived in (agent-scope release); the first wave of
// every workgroup polls all of them, 64 to a load, until none is behind, then
// acquires.  A shared counter instead made the arrivals queue: with the charge's
// adds (below) the barrier took 19300 cycles at 65 workgroups and 4400 at two.
// Every wait is bounded: past spin_limit polls, or once another workgroup has
// given up (word kSmallAbort), the barrier reports failure and the caller
// leaves the kernel.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool grid_barrier(uint32_t* bar, int nblocks, uint32_t& gen, uint32_t spin_limit,
                                             int32_t* okflag) {
    wait_memory();
    __syncthreads();
    ++gen;
    if (threadIdx.x < 64) {
        if (threadIdx.x == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __hip_atomic_store(&bar[blockIdx.x], gen, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        int32_t ok = 1;
        uint32_t n = 0;
        for (;;) {
            bool behind = false;
            for (int b = threadIdx.x; b < nblocks; b += 64)
                behind |= (int32_t)(__hip_atomic_load(&bar[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - gen) < 0;
            if (__ballot(behind) == 0) break;
            if (++n > spin_limit ||
                __hip_atomic_load(&bar[kSmallAbort], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
                ok = 0;
                if (threadIdx.x == 0)
                    __hip_atomic_store(&bar[kSmallAbort], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (threadIdx.x == 0) *okflag = ok;
    }
    __syncthreads();
    return *okflag != 0;
}

// Adds this workgroup's LDS limbs into the device accumulator g (re-split so
// that the device-scope adds never carry, as flush_limbs does) and clears them.
__device__ __forceinline__ void small_flush(u64* __restrict__ acc, int N, u64* __restrict__ g) {
    for (int c = threadIdx.x; c < N; c += blockDim.x) {
        const u128 v = limbs_to_u128(acc[c], acc[N + c], acc[2 * N + c]);
        acc[c] = 0;
        acc[N + c] = 0;
        acc[2 * N + c] = 0;
        const u64 l0 = (u64)v & kLimbMask, l1 = (u64)(v >> 43) & kLimbMask, l2 = (u64)(v >> 86);
        if (l0) __hip_atomic_fetch_add(g + 3 * c, l0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (l1) __hip_atomic_fetch_add(g + 3 * c + 1, l1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (l2) __hip_atomic_fetch_add(g + 3 * c + 2, l2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------
// Gaussian stencils (R = 6, 7): SCHEME 0 leapfrog (src/Gaussian.jl:8-10),
// SCHEME 1 implicit midpoint with the Picard loop
// (src/GaussianFixedPointQuiet.jl:8-10).  Workgroups 0..K-1 hold particles
// (particle p on segment p mod 32K, slot p / 32K); workgroup K computes the
// diagnostics of each step from the velocities the others store.
// ---------------------------------------------------------------------------

// Per-workgroup state of k_small_gauss that is not per particle.
struct GaussCtl {
    int32_t* okflag;  // LDS: the barrier's verdict for the workgroup
    int nblocks;
    uint32_t gen;
    int64_t nb;       // barriers passed: accumulator nb % 3 is filled before barrier nb
    bool diagwg, fit;
    double iN;
};

// Deposit of every held particle's centre (the caller's positions), the
// flush into device accumulator nb % 3, the barrier, and the summed charge
// staged bit-reversed for the solve.  An accumulator is kSmallCopies grids:
// workgroup b adds into grid b % 8 (its own XCD's), so that adds to one word
// queue eight deep and not 64, and the readers sum the grids.  Returns false if
// the barrier failed.
template <int R, int JMAX>
__device__ __forceinline__ bool small_deposit_and_meet(const SmallRun& a, const SmallLds& L, GaussCtl& C,
                                                       const double (&cen)[JMAX], const bool (&has)[JMAX], int e) {
    static_assert(kSmallCopies == 8, "eight lanes sum a cell");
    const InstDesc& I = a.I;
    const int N = I.N;
    const int64_t copy = 3 * (int64_t)N, set = kSmallCopies * copy;
    if (!C.diagwg) {
#pragma unroll
        for (int j = 0; j < JMAX; ++j)
            if (has[j]) seg_deposit<R>(L.acc, N, cen[j], (double)N, C.iN, I.nmask, I.w, I.q, C.fit, e);
        __syncthreads();
        small_flush(L.acc, N, a.gacc + set * (C.nb % 3) + copy * (blockIdx.x % kSmallCopies));
    }
    if (!grid_barrier(a.bar, C.nblocks, C.gen, a.spin_limit, C.okflag)) return false;
    // the accumulator read two barriers ago is free again
    for (int b = blockIdx.x; b < kSmallCopies && !C.diagwg; b += a.K)
        for (int c = threadIdx.x; c < copy; c += blockDim.x)
            st_agent(a.gacc + set * ((C.nb + 2) % 3) + copy * b + c, 0);
    const u64* g = a.gacc + set * (C.nb % 3);
    for (int i = threadIdx.x; i < kSmallCopies * N; i += blockDim.x) {
        const int c = i / kSmallCopies;
        const u64* p = g + copy * (i % kSmallCopies) + 3 * c;
        const u64 l0 = ld_agent(p), l1 = ld_agent(p + 1), l2 = ld_agent(p + 2);
        const u64 s0 = sum8_u64(l0), s1 = sum8_u64(l1), s2 = sum8_u64(l2);
        if (i % kSmallCopies == 0) L.re[(int)brev((uint32_t)c, I.log2N)] = fxp_to(limbs_to_u128(s0, s1, s2), I.q);
    }
    __syncthreads();
    ++C.nb;
    return true;
}

// Diagnostics workgroup, one wave per 4096-particle chunk c: the canonical sums
// of v^2 and v/P of a step that ended before the last barrier, from the
// velocities stored then, into dp.  Tree lane t = l + 64 u folds particles
// t + 256 i in order.
__device__ __forceinline__ void small_chunk_sums(const SmallRun& a, const SmallLds& L, int c, int64_t row,
                                                 int32_t step0) {
    const int64_t P = a.I.P, left = P - (int64_t)c * kTreeChunk;
    const int n = (int)(left < kTreeChunk ? left : kTreeChunk);
    const u64* v = reinterpret_cast<const u64*>(((step0 + row + 1) & 1) ? a.V1 : a.V0) + (int64_t)c * kTreeChunk;
    const int l = threadIdx.x & 63;
    const DivP divP(P);
    double s2[4] = {0.0, 0.0, 0.0, 0.0}, s1[4] = {0.0, 0.0, 0.0, 0.0};
    for (int m0 = 0; 64 * m0 < n; m0 += 16) {  // element l + 64 m, m = u + 4 i
        double x[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int i = l + 64 * (m0 + m);
            x[m] = i < n ? __longlong_as_double((long long)ld_agent(v + i)) : 0.0;
        }
#pragma unroll
        for (int m = 0; m < 16; ++m)
            if (l + 64 * (m0 + m) < n) {
                s2[m & 3] = s2[m & 3] + x[m] * x[m];
                s1[m & 3] = s1[m & 3] + divP(x[m]);
            }
    }
    double r[2] = {(s2[0] + s2[2]) + (s2[1] + s2[3]), (s1[0] + s1[2]) + (s1[1] + s1[3])};
    wave_tree<2>(r, [](int, double p, double q) { return p + q; });
    if (l == 0) {
        L.dp[2 * c] = r[0];
        L.dp[2 * c + 1] = r[1];
    }
}

template <int R, int SCHEME, int E>
__global__ void __launch_bounds__(kSmallThreads)
k_small_gauss(SmallRun a) {
    extern __shared__ double sm[];
    __shared__ int32_t okflag;
    const InstDesc I = a.I;
    const InstState S0 = *a.st;
    const int N = I.N, log2N = I.log2N;
    const SmallLds L = small_lds(sm, N);
    const int K = a.K;
    GaussCtl C;
    C.okflag = &okflag;
    C.nblocks = K + 1;
    C.gen = 0;
    C.nb = 0;
    C.diagwg = (int)blockIdx.x == K;
    C.fit = limbs_fit(I.w, I.q);
    C.iN = 1.0 / (double)N;
    const int e = threadIdx.x & (kSegLanes - 1);
    const int64_t seg = (int64_t)blockIdx.x * kSegs + (threadIdx.x >> 4);
    const int64_t G = (int64_t)K * kSegs;
    const int64_t P = I.P;
    const double Nd = (double)N, dt = I.dt;
    const int32_t nmask = I.nmask;
    constexpr int JMAX = kSmallMaxSlots;
    // particle state: X, V of the step and the Picard iterate v_k
    double Xp[JMAX], Vp[JMAX], vk[JMAX], cen[JMAX];
    bool has[JMAX];
    {
        const int par = S0.step & 1;
        const double* X = par ? a.X1 : a.X0;
        const double* V = par ? a.V1 : a.V0;
#pragma unroll
        for (int j = 0; j < JMAX; ++j) {
            const int64_t p = seg + G * j;
            has[j] = !C.diagwg && p < P;
            Xp[j] = has[j] ? X[p] : 0.0;
            Vp[j] = has[j] ? V[p] : 0.0;
            vk[j] = Vp[j];
            cen[j] = 0.0;
        }
    }
    {
        const double* Ein = S0.e_cur ? a.E1 : a.E0;
        for (int j = threadIdx.x; j < N; j += blockDim.x) {
            L.Fl[j] = Ein[j];
            L.Eld[j] = Ein[j];
        }
    }
    for (int c = threadIdx.x; c < 3 * N; c += blockDim.x) L.acc[c] = 0;
    stage_tables(L, a.tw, N);
    WaveTables<E> W;
    load_wave_tables<E>(W, L, N);
    bool bad = false, ok = true;
    int64_t pend_row = -1;  // diagnostics workgroup: step whose row is still to be written
    int32_t pend_sweeps = 0;
    double pend_se = 0.0;
    const int nch = (int)((P + kTreeChunk - 1) / kTreeChunk);
    // The field of the staged charge (wave 0); in the diagnostics workgroup
    // beside it the sums of the pending step (waves 1..nch) and its row.
    // Returns the convergence test.
    auto solve = [&](auto test) {
        const bool pend = C.diagwg && pend_row >= 0;
        if (threadIdx.x < 64) wave_solve<decltype(test)::value, E>(L, W, N, log2N, I.rtol);
        else if (pend && (int)threadIdx.x < 64 * (1 + nch))
            small_chunk_sums(a, L, (int)(threadIdx.x >> 6) - 1, pend_row, S0.step);
        __syncthreads();
        if (pend && threadIdx.x == 0)
            small_diag_row(L, I, pend_se, nch, a.diag + 4 * pend_row, a.sweeps + pend_row, pend_sweeps);
        pend_row = -1;
        bad = bad || !isfinite(L.red[0]);
        return L.red[1] != 0.0;
    };

    for (int64_t s = 0; s < a.nsteps && ok; ++s) {
        const int paro = (int)((S0.step + s + 1) & 1);
        u64* Xo = reinterpret_cast<u64*>(paro ? a.X1 : a.X0);
        u64* Vo = reinterpret_cast<u64*>(paro ? a.V1 : a.V0);
        if (SCHEME == 0) {
            // u(); deposit at x (centre (x + x)/2)
#pragma unroll
            for (int j = 0; j < JMAX; ++j) {
                Xp[j] = has[j] ? jl_mod1f(Xp[j] + (Vp[j] / 2.0) * dt) : 0.0;
                cen[j] = (Xp[j] + Xp[j]) / 2.0;
            }
            if (!(ok = small_deposit_and_meet<R, JMAX>(a, L, C, cen, has, e))) break;
            solve(std::false_type{});
            pend_se = L.red[2];
            // u(); v += gather(E, x)*dt
#pragma unroll
            for (int j = 0; j < JMAX; ++j)
                if (has[j]) {
                    Xp[j] = jl_mod1f(Xp[j] + (Vp[j] / 2.0) * dt);
                    Vp[j] = Vp[j] + seg_gather<R>(L.Eld, Xp[j], Nd, C.iN, nmask, e) * dt;
                    if (e == 0) {
                        st_agent(Xo + seg + G * j, (u64)__double_as_longlong(Xp[j]));
                        st_agent(Vo + seg + G * j, (u64)__double_as_longlong(Vp[j]));
                    }
                }
            pend_row = s;
            pend_sweeps = 1;
        } else {
            // X .= x; V .= v; the loop's first iterate is v_0 = V:
            // x_0 = X + ((V + V)/2)*dt, centre (x_0 + X)/2
#pragma unroll
            for (int j = 0; j < JMAX; ++j) {
                vk[j] = Vp[j];
                const double x = Xp[j] + ((vk[j] + Vp[j]) / 2.0) * dt;
                cen[j] = (x + Xp[j]) / 2.0;
            }
            if (!(ok = small_deposit_and_meet<R, JMAX>(a, L, C, cen, has, e))) break;
            for (int k = 0;; ++k) {
                const bool conv = solve(std::true_type{});
                const bool done = conv || k == I.max_sweeps - 1;
                // v_{k+1} = V + gather(E_k, c_k)*dt; unless the loop ends here
                // the next centre c_{k+1} = (x_{k+1} + X)/2
#pragma unroll
                for (int j = 0; j < JMAX; ++j)
                    if (has[j]) {
                        const double x = Xp[j] + ((vk[j] + Vp[j]) / 2.0) * dt;
                        const double vn = Vp[j] + seg_gather<R>(L.Eld, (x + Xp[j]) / 2.0, Nd, C.iN, nmask, e) * dt;
                        if (done) {
                            Xp[j] = jl_mod1f(x);
                            Vp[j] = vn;
                            if (e == 0) {
                                st_agent(Xo + seg + G * j, (u64)__double_as_longlong(Xp[j]));
                                st_agent(Vo + seg + G * j, (u64)__double_as_longlong(Vp[j]));
                            }
                        } else {
                            vk[j] = vn;
                            const double x2 = Xp[j] + ((vn + Vp[j]) / 2.0) * dt;
                            cen[j] = (x2 + Xp[j]) / 2.0;
                        }
                    }
                if (done) {
                    pend_row = s;
                    pend_sweeps = k + 1;
                    pend_se = L.red[2];
                    break;
                }
                if (!(ok = small_deposit_and_meet<R, JMAX>(a, L, C, cen, has, e))) break;
            }
        }
    }
    if (ok) ok = grid_barrier(a.bar, C.nblocks, C.gen, a.spin_limit, C.okflag);
    if (ok && C.diagwg && pend_row >= 0) {
        if ((int)threadIdx.x < 64 * nch) small_chunk_sums(a, L, (int)(threadIdx.x >> 6), pend_row, S0.step);
        __syncthreads();
        if (threadIdx.x == 0)
            small_diag_row(L, I, pend_se, nch, a.diag + 4 * pend_row, a.sweeps + pend_row, pend_sweeps);
    }
    if (blockIdx.x == 0 && ok) {
        double* Eo = S0.e_cur ? a.E1 : a.E0;
        for (int j = threadIdx.x; j < N; j += blockDim.x) Eo[j] = L.Eld[j];
        if (threadIdx.x == 0) {
            InstState S = S0;
            S.step += (int32_t)a.nsteps;
            S.last_sweep = -1;
            if (bad) S.err |= 1;
            *a.st = S;
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
bool small_eligible(const InstDesc& I, int scheme, int precision, int64_t* K_out) {
    if (precision != 0 || I.N > kSmallMaxN) return false;
    if (I.R == 0) {
        if (scheme != 0 || I.P > (int64_t)kSmallThreads * kSmallNgpSlots) return false;
        *K_out = 1;
        return true;
    }
    if ((I.R != 6 && I.R != 7) || (scheme != 0 && scheme != 1)) return false;
    // one slot per segment while the particles fill at most kSmallMaxGroups
    // workgroups, then more slots per segment
    int64_t K = (I.P + kSegs - 1) / kSegs;
    if (K > kSmallMaxGroups) K = kSmallMaxGroups;
    if ((I.P + K * kSegs - 1) / (K * kSegs) > kSmallMaxSlots) return false;
    *K_out = K;
    return true;
}

int small_workgroups_ok(const InstDesc& I, int64_t K) {
    if (I.R == 0) return K == 1;
    return K >= 1 && K <= kSmallMaxGroups && (I.P + K * kSegs - 1) / (K * kSegs) <= kSmallMaxSlots;
}

// the kernel of a shape, scheme and solve width
template <int E>
static const void* small_kernel(int R, int scheme) {
    if (R == 0) return reinterpret_cast<const void*>(k_small_ngp<E>);
    if (R == 6)
        return scheme ? reinterpret_cast<const void*>(k_small_gauss<6, 1, E>)
                      : reinterpret_cast<const void*>(k_small_gauss<6, 0, E>);
    return scheme ? reinterpret_cast<const void*>(k_small_gauss<7, 1, E>)
                  : reinterpret_cast<const void*>(k_small_gauss<7, 0, E>);
}

hipError_t launch_small_run(const SmallRun& a, int scheme, hipStream_t s) {
    const unsigned lds = (unsigned)small_lds_bytes(a.I.N);
    SmallRun arg = a;
    void* args[] = {&arg};
    const void* f = a.I.N <= 64 ? small_kernel<1>(a.I.R, scheme)
                                : a.I.N <= 128 ? small_kernel<2>(a.I.R, scheme) : small_kernel<4>(a.I.R, scheme);
    if (a.I.R == 0) return hipLaunchKernel(f, dim3(1), dim3(kSmallThreads), args, lds, s);
    return hipLaunchCooperativeKernel(f, dim3((unsigned)a.K + 1), dim3(kSmallThreads), args, lds, s);
}

int configure_kernels_small() {
    const int bytes = small_lds_bytes(kSmallMaxN);
    hipError_t e = hipSuccess;
    auto chk = [&](hipError_t r) { if (r != hipSuccess) e = r; };
    for (int R : {0, 6, 7})
        for (int scheme = 0; scheme < 2; ++scheme)
            for (const void* f : {small_kernel<1>(R, scheme), small_kernel<2>(R, scheme), small_kernel<4>(R, scheme)})
                chk(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    (void)hipGetLastError();
    return e == hipSuccess ? 0 : -1;
}

}  // namespace pic
