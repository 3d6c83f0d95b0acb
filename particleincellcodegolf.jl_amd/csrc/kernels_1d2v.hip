// kernels_1d2v.hip -- FP64 gfx950 kernels of the magnetised 1D2V step
// (src/NGP1D2V.jl, src/NGP1D2V2S.jl): explicit Boris push with the Gaussian
// stencil, one or two species, and the time-binned field.  Compiled with
// -ffp-contract=off: results are bitwise equal to the CPU restatement.
//
// Per step: the solve reads the exact signed charge deposited by the previous
// push (or by the prime deposit after an upload), writes E, adds it into its
// time bin and sums E^2; the push gathers E at x, applies the Boris rotation,
// moves and wraps the particle and deposits its charge for the next step; the
// diagnostics (predicated on t % bin == 0) sum the kinetic terms and write a
// row of D, and advance the step counter.
#include "pic1d2v_internal.h"
#include "pic_device.h"
#include "seg16.h"
#include "solve1d.h"
#include "stencil1d.h"
#include "wave_fft.h"

#pragma clang fp contract(off)

namespace pic {

// r[k[1]] += q*k[2]*w over d(c) (src/NGP1D2V2S.jl:28): each contribution's
// magnitude on the 2^-qb grid into the LDS limbs of the species' sign.
template <int R>
__device__ __forceinline__ void deposit_gauss_q(u64* __restrict__ acc, int32_t N, double c, double Nd,
                                                int32_t nmask, double q, double w, int qb) {
    const double cN = c * Nd, i0d = rint(cN);
    if (!edges_fit(cN) || !limbs_fit(q * w, qb)) {
        const int64_t i0 = (int64_t)i0d;
        double prev = edge_half_erf(i0 - R, c, Nd);
#pragma unroll 1
        for (int j = -R; j <= R; ++j) {
            const double next = edge_half_erf(i0 + j + 1, c, Nd);
            const double wt = next - prev;
            prev = next;
            const double a = (q * wt) * w;
            if (a != 0.0) lds_add_fxp(acc, N, cell0(i0 + j, nmask), fxp_from(fabs(a), qb));
        }
        return;
    }
    double f[2 * R + 2];
    gauss_edges<R>(c, i0d, Nd, 1.0 / Nd, f);
    const int32_t i0 = (int32_t)(int64_t)i0d;
#pragma unroll
    for (int j = -R; j <= R; ++j) {
        if (j == -7 || j == 7) continue;  // both edges beyond 6: the weight is exactly 0
        const double wt = f[j + R + 1] - f[j + R];
        lds_add_contribution(acc, N, (i0 + j - 1) & nmask, (q * wt) * w, qb);
    }
}

// boris(vx, vy, E, B, dt, q_m) of src/NGP1D2V2S.jl:5-11 with every product of
// the SVector cross products made, zeros included; q_m = 1 is
// src/NGP1D2V.jl:5-10 (E*dt/2 == E*(dt/2)).
__device__ __forceinline__ void boris12(double& vx, double& vy, double E, double B, double dt, double q_m) {
    const double h = (dt / 2.0) * q_m;
    const double m1 = vx + E * h, m2 = vy, m3 = 0.0;
    const double t1 = 0.0, t2 = 0.0, t3 = B * h;
    const double c1 = m2 * t3 - m3 * t2, c2 = m3 * t1 - m1 * t3, c3 = m1 * t2 - m2 * t1;
    const double a1 = m1 + c1, a2 = m2 + c2, a3 = m3 + c3;
    const double d1 = a2 * t3 - a3 * t2, d2 = a3 * t1 - a1 * t3;
    const double s = 1.0 + ((t1 * t1 + t2 * t2) + t3 * t3);
    vx = (m1 + (2.0 * d1) / s) + E * h;
    vy = m2 + (2.0 * d2) / s;
}

// The charge of every tile's particles at their current positions.
template <int R>
__global__ void __launch_bounds__(1024)
k12_deposit(const Tile12* __restrict__ tiles, const double* __restrict__ x, u64* __restrict__ racc, int N,
            double q0, double q1, double w, int qb) {
    extern __shared__ u64 lds[];
    const Tile12 T = tiles[blockIdx.x];
    const double q = T.species ? q1 : q0;
    zero_lds(lds, 3 * N);
    __syncthreads();
    const double Nd = (double)N;
    for (int64_t p = threadIdx.x; p < T.count; p += blockDim.x)
        deposit_gauss_q<R>(lds, N, x[T.start + p], Nd, N - 1, q, w, qb);
    __syncthreads();
    flush_limbs(lds, N, racc + (q < 0.0 ? 3 * N : 0));
}

// E = real(ifft(fft(rho) ./ ik)) from the exact signed charge (which it
// clears), Es[:, ceil(t/bin)] .+= E and sum(abs2, E).  One block.
// Mixed (racc32 set): the charge is per species u64 quanta, cq[s] each
// (q_s * w * 2^-30), summed in FP64; E32 gets E * escale2 in FP32.
__global__ void __launch_bounds__(kSolveThreads)
k12_solve(u64* __restrict__ racc, double* __restrict__ E, double* __restrict__ Es, int64_t cap_bins,
          State12* __restrict__ st, const double2* __restrict__ twp, int N, int log2N, int qb, int bin,
          u64* __restrict__ racc32, double cq0, double cq1, float* __restrict__ E32, double escale2) {
    extern __shared__ double sm[];
    const int NP = solve_np(N);
    double* re = sm;
    double* im = sm + NP;
    double* red = sm + 2 * NP + N;
    SolveRegs Rg;
    solve_prefetch(Rg, twp, N, log2N);
    for (int j = threadIdx.x; j < N; j += blockDim.x) {
        double r;
        if (racc32) {
            const u64 a0 = racc32[j], a1 = racc32[N + j];
            racc32[j] = 0;
            racc32[N + j] = 0;
            r = cq0 * (double)a0 + cq1 * (double)a1;
        } else {
            u64* a = racc + 3 * j;
            u64* b = racc + 3 * N + 3 * j;
            const u128 pos = limbs_to_u128(a[0], a[1], a[2]), neg = limbs_to_u128(b[0], b[1], b[2]);
            a[0] = 0;
            a[1] = 0;
            a[2] = 0;
            b[0] = 0;
            b[1] = 0;
            b[2] = 0;
            r = pos >= neg ? fxp_to(pos - neg, qb) : -fxp_to(neg - pos, qb);
        }
        const int k = padi((int)brev((uint32_t)j, log2N));
        re[k] = r;
        im[k] = 0.0;
    }
    __syncthreads();
    solve_lds(re, im, Rg, twp, N, log2N);
    const int64_t t = st->step + 1;
    const int64_t bi = (t + bin - 1) / bin - 1;
    for (int j = threadIdx.x; j < N; j += blockDim.x) {
        const double e = solve_at(re, j);
        E[j] = e;
        if (E32) E32[j] = (float)(e * escale2);
        if (bi < cap_bins) Es[bi * N + j] = Es[bi * N + j] + e;
    }
    const double se = block_chunk_sum(red, N, [&](int64_t i) {
        const double e = solve_at(re, (int)i);
        return e * e;
    });
    const double emax = block_maxabs(red, N, [&](int64_t i) { return solve_at(re, (int)i); });
    if (threadIdx.x == 0) {
        st->se = se;
        if (!isfinite(emax)) st->err |= 1;
    }
}

// Ej = sum(k->E[k[1]]*k[2], d(x[j])); (vx, vy) = boris(...); x = mod(x + vx*dt, 1);
// then the particle's charge at the new x for the next step.
template <int R>
__global__ void __launch_bounds__(1024)
k12_push(const Tile12* __restrict__ tiles, double* __restrict__ x, double* __restrict__ vx,
         double* __restrict__ vy, const double* __restrict__ E, u64* __restrict__ racc, int N, double q0,
         double q1, double qm0, double qm1, double w, int qb, double B0, double dt) {
    extern __shared__ u64 lds[];
    const Tile12 T = tiles[blockIdx.x];
    const double q = T.species ? q1 : q0, qm = T.species ? qm1 : qm0;
    double* Eld = reinterpret_cast<double*>(lds);
    u64* acc = lds + N;
    for (int i = threadIdx.x; i < N; i += blockDim.x) Eld[i] = E[i];
    zero_lds(acc, 3 * N);
    __syncthreads();
    const double Nd = (double)N;
    const int32_t nmask = N - 1;
    for (int64_t p = threadIdx.x; p < T.count; p += blockDim.x) {
        const int64_t g = T.start + p;
        const double xj = x[g];
        double u = vx[g], v = vy[g];
        const double Ej = gather_gauss<R>(Eld, xj, Nd, nmask);
        boris12(u, v, Ej, B0, dt, qm);
        const double xn = jl_mod1f(xj + u * dt);
        x[g] = xn;
        vx[g] = u;
        vy[g] = v;
        deposit_gauss_q<R>(acc, N, xn, Nd, nmask, q, w, qb);
    }
    __syncthreads();
    flush_limbs(acc, N, racc + (q < 0.0 ? 3 * N : 0));
}

// Diagnostics partials over chunk c of 4096 particle indices:
// sum(vy^2 + vx^2 [+ M*(vy2^2 + vx2^2)]), sum(vx/P [+ M*vx2/P]), same for vy.
// red: LDS of 4*kTreeLanes + 8 doubles; every thread of the block calls.
__device__ __forceinline__ void diag_chunk12(double* red, const double* vx, const double* vy, int64_t P, int ns,
                                             double m0, double m1, int64_t chunk, double* dpart) {
    const int64_t s = chunk * kTreeChunk;
    const int64_t n = P - s < kTreeChunk ? P - s : kTreeChunk;
    const double Pd = (double)P;
    double a = 0.0, b = 0.0, c = 0.0;
    if (threadIdx.x < kTreeLanes)
        for (int64_t i = threadIdx.x; i < n; i += kTreeLanes) {
            const int64_t j = s + i;
            const double x0 = vx[j], y0 = vy[j];
            double k = m0 * ((y0 * y0) + (x0 * x0));
            double mx = (m0 * x0) / Pd, my = (m0 * y0) / Pd;
            if (ns == 2) {
                const double x1 = vx[P + j], y1 = vy[P + j];
                k = k + m1 * ((y1 * y1) + (x1 * x1));
                mx = mx + (m1 * x1) / Pd;
                my = my + (m1 * y1) / Pd;
            }
            a = a + k;
            b = b + mx;
            c = c + my;
        }
    tree256x3<false>(red, a, b, c);
    if (threadIdx.x == 0) {
        dpart[0] = a;
        dpart[1] = b;
        dpart[2] = c;
    }
}

// the partials when t % bin == 0
__global__ void __launch_bounds__(256)
k12_diag_chunks(const double* __restrict__ vx, const double* __restrict__ vy, int64_t P, int ns, double m0,
                double m1, int bin, const State12* __restrict__ st, double* __restrict__ dpart) {
    __shared__ double red[4 * kTreeLanes + 8];
    if ((st->step + 1) % bin != 0) return;
    diag_chunk12(red, vx, vy, P, ns, m0, m1, blockIdx.x, dpart + 3 * blockIdx.x);
}

// Canonical tree over n values spread with stride 3 (in place).
__device__ double tree_stride3(double* red, double* vals, int64_t n) {
    while (n > kTreeChunk) {
        const int64_t C = (n + kTreeChunk - 1) / kTreeChunk;
        for (int64_t c = 0; c < C; ++c) {
            const int64_t m = n - c * kTreeChunk < kTreeChunk ? n - c * kTreeChunk : kTreeChunk;
            const double s = block_chunk_sum(red, m, [&](int64_t i) { return vals[3 * (c * kTreeChunk + i)]; });
            if (threadIdx.x == 0) vals[3 * c] = s;
            __syncthreads();
        }
        n = C;
    }
    return block_chunk_sum(red, n, [&](int64_t i) { return vals[3 * i]; });
}

// D[t/bin, 1:5] (src/NGP1D2V2S.jl:52-56) of step t, t % bin == 0, from the
// chunk partials; every thread of the block calls.
__device__ void diag_row12(double* red, double* dpart, int64_t nchunks, int64_t P, int N, double n0, int bin, int64_t t,
                           double se, double* D, int64_t cap_bins) {
    const double sk = tree_stride3(red, dpart, nchunks);
    const double sx = tree_stride3(red, dpart + 1, nchunks);
    const double sy = tree_stride3(red, dpart + 2, nchunks);
    const int64_t bi = t / bin - 1;
    if (threadIdx.x == 0 && bi < cap_bins) {
        double* row = D + 5 * bi;
        row[0] = row[0] + (se / (double)N) / 2.0;
        row[1] = row[1] + ((sk * n0) / (double)P) / 2.0;
        row[3] = row[3] + sx;
        row[4] = row[4] + sy;
        row[2] = row[2] + (row[0] + row[1]);
        for (int c = 0; c < 3; ++c) row[c] = row[c] * (2.0 / n0);
    }
}

// the row when t % bin == 0; then step += 1.
__global__ void __launch_bounds__(256)
k12_diag_final(double* __restrict__ dpart, int64_t nchunks, int64_t P, int N, double n0, int bin,
               State12* __restrict__ st, double* __restrict__ D, int64_t cap_bins) {
    __shared__ double red[kTreeLanes + 8];
    const int64_t t = st->step + 1;
    if (t % bin == 0) diag_row12(red, dpart, nchunks, P, N, n0, bin, t, st->se, D, cap_bins);
    if (threadIdx.x == 0) st->step = t;
}

// ---------------------------------------------------------------------------
// The FP64 step at the scripts' sizes (N <= kSmallN12, ns*P <= kSmallP12) in one
// launch.  At some thousand particles the general chain's four launches are
// latency: a push walks a particle's two stencils in one thread (15 us), the
// solve is one block's LDS passes (10 us), and the two diagnostics launches
// mostly end at their first test (2 x 4.5 us).  Here a particle takes a row of 16
// lanes, and every block solves the field for itself in its first wave
// (wave_fft.h) while the others evaluate their first particles' gather weights:
// the launch boundary is the only meeting of the blocks.  Buffers that a launch
// both reads and writes take turns: three charge accumulators (read, added to,
// cleared) and two copies of the velocities, so that block 0, which has no
// particles, can sum the velocities of the step before while this one's are
// written.  The turn is the step number mod kSmallTurns12, known to the host.
//
// A chain of latencies bounds it: launch 3 us, loads 2, solve 4, fold and Boris
// 0.6, the new stencil 1.6, adds 0.7.  2 x 2048 particles on 256 cells: 27.1 us a
// step in the general chain, 13.4 here; 18.4 with the solve and the row in the
// last block to arrive.  Every block adds its grid to the same words, and more
// waves in a block run their erf chains in turn: 32 particles a block 13.4 us,
// 16 15.1, 48 13.6.
// ---------------------------------------------------------------------------

// E of the charge in sm (bit-reversed) into Eld, by a block's first wave, whose
// lanes return their elements too.  sm: 3N doubles.
template <int E>
__device__ __forceinline__ void small_solve12(const double2* tw, int N, int log2N, double* sm,
                                              double* Eld, double (&x)[E]) {
    const int l = threadIdx.x & 63;
    double* line = sm;
    double* pr = sm + N;  // re, im
    if (threadIdx.x >= 64) return;
    const double* xi = reinterpret_cast<const double*>(tw) + kXiOffset;
    double2 w6[6];
    load_wave_twiddles(w6, tw, N);
    double re[E], im[E], xt[E];
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int m = q * 64 + l;
        re[q] = m < N ? line[m] : 0.0;
        im[q] = 0.0;
        xt[q] = m >= N ? 0.0 : m == 0 ? xi[1] : (m <= N / 2 ? xi[m] : -xi[N - m]);
    }
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {  // one copy of the transform's code: it is fetched anew by each launch
        wave_radix2<E>(re, im, w6, tw, N, pass != 0);
        if (pass) break;
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int m = q * 64 + l;
            if (m >= N) continue;
            double a = im[q] * xt[q];
            double b = -(re[q] * xt[q]);
            if (m == 0) {
                a = a * 0.0;
                b = b * 0.0;
            }
            const int p = (int)brev((uint32_t)m, log2N);
            pr[p] = a;
            pr[N + p] = b;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int i = q * 64 + l;
            re[q] = i < N ? pr[i] : 0.0;
            im[q] = i < N ? pr[N + i] : 0.0;
        }
    }
    const double scale = 1.0 / (double)N;
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int i = q * 64 + l;
        x[q] = i < N ? re[q] * scale : 0.0;
        if (i < N) Eld[i] = x[q];
    }
}

// the D row of step t from the velocities after it, by a whole block
__device__ void small_row12(const Buffers12& b, double* sm, int64_t t, double se, const double* vx, const double* vy) {
    for (int64_t c = 0; c < b.nchunks; ++c) {
        diag_chunk12(sm, vx, vy, b.P, b.ns, b.mass[0], b.mass[1], c, b.dpart + 3 * c);
        __syncthreads();
    }
    diag_row12(sm, b.dpart, b.nchunks, b.P, b.N, b.n0, b.bin, t, se, b.D, b.cap_bins);
    __syncthreads();
}

template <int R, int E>
__global__ void __launch_bounds__(kSmallThreads12 + 64) k12_small_step(Buffers12 b, int turn) {
    extern __shared__ double sm[];
    static_assert(kSmallThreads12 + 64 >= kTreeLanes, "the row's trees");
    constexpr int kSegs = kSmallThreads12 / kSegLanes;
    const int N = b.N, e = threadIdx.x & (kSegLanes - 1);
    double* Eld = sm;                                 // N
    u64* acc = reinterpret_cast<u64*>(sm + N);        // the positive charge's limbs, then the negative's
    double* line = sm + 7 * N;                        // 3N
    const int64_t all = b.ns * b.P;
    const double *vx0 = b.vx + (turn & 1) * all, *vy0 = b.vy + (turn & 1) * all;
    double *vx1 = b.vx + (1 - (turn & 1)) * all, *vy1 = b.vy + (1 - (turn & 1)) * all;
    u64* racc = (u64*)b.racc;
    const u64* rd = racc + 6 * N * (turn % 3);
    u64* add = racc + 6 * N * ((turn + 1) % 3);
    u64* clr = racc + 6 * N * ((turn + 2) % 3);
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
        const u128 pos = limbs_to_u128(rd[3 * i], rd[3 * i + 1], rd[3 * i + 2]),
                   neg = limbs_to_u128(rd[3 * N + 3 * i], rd[3 * N + 3 * i + 1], rd[3 * N + 3 * i + 2]);
        line[(int)brev((uint32_t)i, b.log2N)] = pos >= neg ? fxp_to(pos - neg, b.qbits) : -fxp_to(neg - pos, b.qbits);
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 6 * N; i += gridDim.x * blockDim.x) clr[i] = 0;
    zero_lds(acc, 6 * N);
    __syncthreads();
    double x[E];
    if (blockIdx.x == 0) {
        const int64_t done = b.st->step;
        const double se = b.st->se;
        __syncthreads();  // read by all before lane 0 writes them
        small_solve12<E>(b.tw, N, b.log2N, line, Eld, x);
        if (threadIdx.x < 64) {
            const int64_t bi = (done + b.bin) / b.bin - 1;  // of step done + 1
            double y[2][E], r[2];
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int i = q * 64 + threadIdx.x;
                if (i < N && bi < b.cap_bins) b.Es[bi * N + i] = b.Es[bi * N + i] + x[q];
                y[0][q] = fabs(x[q]);
                y[1][q] = x[q] * x[q];
            }
            wave_canon<2, E>(r, y, [](int k, double a, double c) { return k < 1 ? nanmax(a, c) : a + c; });
            if (threadIdx.x == 0) {
                b.st->se = r[1];
                if (!isfinite(r[0])) b.st->err |= 1;
                b.st->step = done + 1;
            }
        }
        if (done > 0 && done % b.bin == 0 && b.st->row != done) {
            __syncthreads();
            small_row12(b, sm, done, se, vx0, vy0);
            if (threadIdx.x == 0) b.st->row = done;
        }
        return;
    }
    const double Nd = (double)N, iN = 1.0 / Nd;
    const int64_t g0 = (int64_t)(blockIdx.x - 1) * kSegs + ((int)threadIdx.x >> 4) - 4;
    const int64_t gs = (int64_t)(gridDim.x - 1) * kSegs;
    double wt = 0.0, xj = 0.0;
    int32_t first = 0;
    if (threadIdx.x < 64) {
        small_solve12<E>(b.tw, N, b.log2N, line, Eld, x);
    } else if (g0 < all) {
        xj = b.x[g0];
        wt = seg_weight<R>(xj, Nd, iN, e, first, N - 1);
    }
    __syncthreads();
    if (threadIdx.x >= 64) {
        for (int64_t g = g0; g < all; g += gs) {
            const int s = g >= b.P ? 1 : 0;
            const double q = b.q[s];
            double u = vx0[g], v = vy0[g];
            if (g != g0) {
                xj = b.x[g];
                wt = seg_weight<R>(xj, Nd, iN, e, first, N - 1);
            }
            const double Ej = seg_fold<R>(Eld[(first + e) & (N - 1)] * wt);
            boris12(u, v, Ej, b.B0, b.dt, b.q_m[s]);
            const double xn = jl_mod1f(xj + u * b.dt);
            if (e == 0) {
                b.x[g] = xn;
                vx1[g] = u;
                vy1[g] = v;
            }
            int32_t to;
            const double a = (q * seg_weight<R>(xn, Nd, iN, e, to, N - 1)) * b.w;
            if (e <= 2 * R && fabs(a) > 0.0) {  // NaN adds nothing
                const int32_t cell = (to + e) & (N - 1);
                u64* r = acc + (q < 0.0 ? 3 * N : 0);
                if (limbs_fit(q * b.w, b.qbits)) lds_add_contribution(r, N, cell, a, b.qbits);
                else lds_add_fxp(r, N, cell, fxp_from(fabs(a), b.qbits));
            }
        }
    }
    __syncthreads();
    flush_limbs(acc, N, add);
    flush_limbs(acc + 3 * N, N, add + 3 * N);
}

// The row of the last step of a run, where its bin is full.
__global__ void __launch_bounds__(256) k12_small_row(Buffers12 b, int turn) {
    __shared__ double sm[4 * kTreeLanes + 8];
    const int64_t done = b.st->step, all = b.ns * b.P;
    small_row12(b, sm, done, b.st->se, b.vx + (turn & 1) * all, b.vy + (turn & 1) * all);
    if (threadIdx.x == 0) b.st->row = done;
}

// rho from the exact signed charge (clearing it), for the deposit operator.
__global__ void k12_rho(u64* __restrict__ racc, double* __restrict__ rho, int N, int qb) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= N) return;
    u64* a = racc + 3 * j;
    u64* b = racc + 3 * N + 3 * j;
    const u128 pos = limbs_to_u128(a[0], a[1], a[2]), neg = limbs_to_u128(b[0], b[1], b[2]);
    a[0] = 0;
    a[1] = 0;
    a[2] = 0;
    b[0] = 0;
    b[1] = 0;
    b[2] = 0;
    rho[j] = pos >= neg ? fxp_to(pos - neg, qb) : -fxp_to(neg - pos, qb);
}

template <int R>
__global__ void __launch_bounds__(256)
k12_op_gather(const double* __restrict__ E, const double* __restrict__ x, int64_t n, double* __restrict__ Ej,
              int N) {
    extern __shared__ double Eld[];
    for (int i = threadIdx.x; i < N; i += blockDim.x) Eld[i] = E[i];
    __syncthreads();
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) Ej[j] = gather_gauss<R>(Eld, x[j], (double)N, N - 1);
}

__global__ void k12_op_boris(double* __restrict__ vx, double* __restrict__ vy, const double* __restrict__ Ej,
                             int64_t n, double B, double dt, double q_m) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    double u = vx[j], v = vy[j];
    boris12(u, v, Ej[j], B, dt, q_m);
    vx[j] = u;
    vy[j] = v;
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
template <int E>
static void small12(const Buffers12& b, int turn, hipStream_t s) {
    const int64_t segs = kSmallThreads12 / kSegLanes, want = (b.ns * b.P + segs - 1) / segs;
    const unsigned nb = 1 + (unsigned)(want < kSmallBlocks12 ? want : kSmallBlocks12);
    const int words = 10 * b.N > 4 * kTreeLanes + 8 ? 10 * b.N : 4 * kTreeLanes + 8;  // the step's; the trees'
    if (b.R == 6) k12_small_step<6, E><<<nb, kSmallThreads12 + 64, 8 * words, s>>>(b, turn);
    else k12_small_step<7, E><<<nb, kSmallThreads12 + 64, 8 * words, s>>>(b, turn);
}
void launch12_small(const Buffers12& b, int turn, hipStream_t s) {
    if (b.N <= 64) small12<1>(b, turn, s);
    else if (b.N <= 128) small12<2>(b, turn, s);
    else if (b.N <= 256) small12<4>(b, turn, s);
    else small12<8>(b, turn, s);
}
void launch12_small_row(const Buffers12& b, int turn, hipStream_t s) { k12_small_row<<<1, 256, 0, s>>>(b, turn); }

int push12_lds_bytes(int N) { return 32 * N; }  // E + three limb arrays

void launch12_deposit(const Buffers12& b, hipStream_t s) {
    if (b.precision == 1) return launch12_deposit32(b, s);
    const int lds = 24 * b.N;
    u64* r = (u64*)b.racc;
    if (b.R == 6)
        k12_deposit<6><<<b.ntiles, b.block, lds, s>>>(b.tiles, b.x, r, b.N, b.q[0], b.q[1], b.w, b.qbits);
    else
        k12_deposit<7><<<b.ntiles, b.block, lds, s>>>(b.tiles, b.x, r, b.N, b.q[0], b.q[1], b.w, b.qbits);
}

void launch12_solve(const Buffers12& b, hipStream_t s) {
    const int lds = solve_lds_doubles(b.N) * 8;
    const bool m = b.precision == 1;
    const double cq0 = m ? b.q[0] * b.w * 0x1p-30 : 0.0, cq1 = m ? b.q[1] * b.w * 0x1p-30 : 0.0;
    k12_solve<<<1, kSolveThreads, lds, s>>>((u64*)b.racc, b.E, b.Es, b.cap_bins, b.st, b.tw, b.N, b.log2N,
                                            b.qbits, b.bin, m ? (u64*)b.racc32 : nullptr, cq0, cq1,
                                            m ? b.E32 : nullptr, b.escale2);
}

void launch12_push(const Buffers12& b, hipStream_t s) {
    if (b.precision == 1) return launch12_push32(b, s);
    const int lds = push12_lds_bytes(b.N);
    u64* r = (u64*)b.racc;
    if (b.R == 6)
        k12_push<6><<<b.ntiles, b.block, lds, s>>>(b.tiles, b.x, b.vx, b.vy, b.E, r, b.N, b.q[0], b.q[1],
                                                   b.q_m[0], b.q_m[1], b.w, b.qbits, b.B0, b.dt);
    else
        k12_push<7><<<b.ntiles, b.block, lds, s>>>(b.tiles, b.x, b.vx, b.vy, b.E, r, b.N, b.q[0], b.q[1],
                                                   b.q_m[0], b.q_m[1], b.w, b.qbits, b.B0, b.dt);
}

void launch12_diag(const Buffers12& b, hipStream_t s) {
    if (b.precision == 1) return launch12_diag32(b, s);
    k12_diag_chunks<<<(unsigned)b.nchunks, 256, 0, s>>>(b.vx, b.vy, b.P, b.ns, b.mass[0], b.mass[1], b.bin,
                                                       b.st, b.dpart);
    k12_diag_final<<<1, 256, 0, s>>>(b.dpart, b.nchunks, b.P, b.N, b.n0, b.bin, b.st, b.D, b.cap_bins);
}

void launch12_rho(const Buffers12& b, double* rho, hipStream_t s) {
    k12_rho<<<(b.N + 255) / 256, 256, 0, s>>>((u64*)b.racc, rho, b.N, b.qbits);
}

void launch12_op_gather(const Buffers12& b, const double* E, const double* x, int64_t n, double* Ej,
                        hipStream_t s) {
    const unsigned g = (unsigned)((n + 255) / 256);
    if (b.R == 6) k12_op_gather<6><<<g, 256, 8 * b.N, s>>>(E, x, n, Ej, b.N);
    else k12_op_gather<7><<<g, 256, 8 * b.N, s>>>(E, x, n, Ej, b.N);
}

void launch12_op_boris(double* vx, double* vy, const double* Ej, int64_t n, double B, double dt, double q_m,
                       hipStream_t s) {
    k12_op_boris<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(vx, vy, Ej, n, B, dt, q_m);
}

template <typename K>
static hipError_t allow12(K kernel, int bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               bytes);
}

int configure_kernels_1d2v() {
    const int big = 32 * kMaxN;
    hipError_t e = hipSuccess;
    auto chk = [&](hipError_t r) { if (r != hipSuccess) e = r; };
    chk(allow12(k12_deposit<6>, big));
    chk(allow12(k12_deposit<7>, big));
    chk(allow12(k12_push<6>, big));
    chk(allow12(k12_push<7>, big));
    chk(allow12(k12_solve, big));
    (void)hipGetLastError();
    return e == hipSuccess ? 0 : -1;
}

}  // namespace pic
