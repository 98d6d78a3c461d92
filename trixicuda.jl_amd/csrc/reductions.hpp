// reductions.hpp -- the device reductions of the callbacks: max_dt, integrals,
// error norms, counts.  Each is one launch: every block leaves a partial, and
// the last block to arrive combines them in a fixed order and writes the result
// (to pinned host memory where the caller waits for it), so that the result
// does not depend on the order of arrival.
//
// Before, one thread added up to 1024 partials (66 us a call) in a launch of
// its own and a copy brought the result back; one thread per element walked its
// nodes (128 blocks at 32768 elements), and the error norms re-read all nodes of
// the element for each analysis point.  3D Euler, 4096 elements: error norms
// 2950 us, integrals 104, max_dt 23; at 32768 elements max_dt 47 + 13.
#pragma once

#include "arrival.hpp"
#include "initial_conditions.hpp"
#include "physics.hpp"

namespace trixi_hip {

// A partial of this block.  Partials and the arrival count cross the XCDs' L2
// caches, so they are accessed at device scope (past the L2) and ordered by
// waiting for the stores; a device-scope fence instead writes back the whole
// L2 once per block, with the state a Runge-Kutta step has just left there
// (max_dt after a step of 32768 elements of 3D Euler: +50 us).
__device__ __forceinline__ void store_partial(double* p, double x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Combines the blocks' partial vectors (m components, the first nsum summed,
// the others their maximum) in the last block to arrive, which writes `out`; the
// count in `arrived` wraps to zero there (arrival.hpp).  Every thread of every
// block calls it after its block's store_partial calls.
// Returns true in the last block's thread 0, with component 0 in `first`.
template <int THREADS>
__device__ __forceinline__ bool finish_partials(const double* partial, double* out, unsigned* arrived, int m,
                                                int nsum, double& first) {
    __shared__ bool last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partials have arrived
    __syncthreads();
    if (threadIdx.x == 0)
        last = arrival_is_last(atomicInc(arrived, gridDim.x - 1), gridDim.x);
    __syncthreads();
    if (!last) return false;
    asm volatile("" ::: "memory");
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    for (int c = wave; c < m; c += THREADS / 64) {
        const bool sum = c < nsum;
        double x = 0.0;  // the maxima are of values >= 0
        // eight loads in flight (each goes past the caches: one at a time they
        // were most of a call)
        for (int b0 = lane; b0 < (int)gridDim.x; b0 += 64 * 8) {
            double y[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int b = b0 + 64 * i;
                y[i] = b < (int)gridDim.x ? __hip_atomic_load(&partial[(int64_t)b * m + c], __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT)
                                          : 0.0;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) x = sum ? x + y[i] : fmax(x, y[i]);
        }
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) {
            const double y = __shfl_xor(x, w);
            x = sum ? x + y : fmax(x, y);
        }
        if (lane == 0) out[c] = x;
        if (c == 0) first = x;
    }
    return threadIdx.x == 0;
}
template <int THREADS>
__device__ __forceinline__ void finish_partials(const double* partial, double* out, unsigned* arrived, int m,
                                                int nsum) {
    double first = 0.0;
    finish_partials<THREADS>(partial, out, arrived, m, nsum, first);
}

// The time loop on the device: the stage times of the CarpenterKennedy2N54 step
// from the current time, time = {stage time, dt} x 5, then {t, done}.  A step of
// size h is shortened to end at t_end (select_step's rule, the same operations
// in the same order); once t has reached t_end every further step sets `done`,
// which the stages read.  log takes {t after the step, h}, h < 0 for no step.
constexpr int TIME_T = 10, TIME_DONE = 11, TIME_DOUBLES = 16;
struct StepControl {
    double* time;  // nullptr: a reduction only
    double* log;   // pinned
    double t_end, cfl;
    int N;
    double c[5];
};
__device__ __forceinline__ void next_step(const StepControl& q, double h) {
    // (no fused multiply-adds but the stage times', which set_time_kernel fuses:
    // the times equal a host loop's bit for bit)
#pragma clang fp contract(off)
    const double t = q.time[TIME_T];
    if (!(t < q.t_end)) {
        q.time[TIME_DONE] = 1.0;
        q.log[0] = t;
        q.log[1] = -1.0;
        return;
    }
    double tn = t + h;
    if (tn >= q.t_end) {
        h = q.t_end - t;
        tn = q.t_end;
    }
    for (int s = 0; s < 5; ++s) {
        q.time[2 * s] = fma(q.c[s], h, t);
        q.time[2 * s + 1] = h;
    }
    q.time[TIME_T] = tn;
    q.log[0] = tn;
    q.log[1] = h;
}
// 2 / (N max) of the largest scaled wave speed
__host__ __device__ inline double max_dt_of(int N, double m) {
    const double tiny = 4.9406564584124654e-324;  // nextafter(0, 1)
    if (!(m > tiny)) m = tiny;
    return 2.0 / (N * m);
}
__global__ void start_time_kernel(double* time, double t) {
    time[TIME_T] = t;
    time[TIME_DONE] = 0.0;
}
__global__ void next_step_kernel(StepControl q, double dt) { next_step(q, dt); }

// Elements per pass of a block and threads of the element reductions: 16
// consecutive elements (whole 128-byte rows of an FP64 state) by 16 groups that
// share an element's nodes.
constexpr int RED_ELEMS = 16, RED_THREADS = 256, RED_GROUPS = RED_THREADS / RED_ELEMS;

// max over elements of invJ_e * sum_d max over nodes |lambda_d|: the largest of
// each direction over the element's nodes, then the sum (Trixi's max_dt).
template <class EQ, int DIM, typename S>
__global__ void __launch_bounds__(RED_THREADS) max_speed_kernel(const S* __restrict__ u,
                                                                const double* __restrict__ invJ,
                                                                double* __restrict__ partial, double* out,
                                                                unsigned* arrived, int nn, int64_t E,
                                                                PhysParams phys, StepControl step) {
    __shared__ double red[RED_THREADS / 64][DIM][RED_ELEMS];
    const PhysR<double> P = PhysR<double>::from(phys);
    const int c = threadIdx.x % RED_ELEMS, g = threadIdx.x / RED_ELEMS;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    double best = 0.0;
    for (int64_t e0 = (int64_t)blockIdx.x * RED_ELEMS; e0 < E; e0 += (int64_t)gridDim.x * RED_ELEMS) {
        const int64_t e = e0 + c < E ? e0 + c : E - 1;
        double lmax[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) lmax[d] = 0.0;
#pragma unroll 4
        for (int n = g; n < nn; n += RED_GROUPS) {
            double uc[EQ::NV], lam[3];
#pragma unroll
            for (int v = 0; v < EQ::NV; ++v) uc[v] = (double)u[((int64_t)v * nn + n) * E + e];
            EQ::max_abs_speeds(uc, P, lam);
#pragma unroll
            for (int d = 0; d < DIM; ++d) lmax[d] = lam[d] > lmax[d] ? lam[d] : lmax[d];
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            lmax[d] = fmax(lmax[d], __shfl_xor(lmax[d], 16));
            lmax[d] = fmax(lmax[d], __shfl_xor(lmax[d], 32));
            if (lane < RED_ELEMS) red[wave][d][lane] = lmax[d];
        }
        __syncthreads();
        if (threadIdx.x < RED_ELEMS) {
            double s = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                double x = red[0][d][c];
#pragma unroll
                for (int w = 1; w < RED_THREADS / 64; ++w) x = fmax(x, red[w][d][c]);
                s += x;
            }
            const double sc = invJ[e] * s;
            best = sc > best ? sc : best;
        }
        __syncthreads();
    }
    if (threadIdx.x < 64) {
#pragma unroll
        for (int w = 8; w > 0; w >>= 1) best = fmax(best, __shfl_xor(best, w));
        if (threadIdx.x == 0) store_partial(&partial[blockIdx.x], best);
    }
    double m = 0.0;
    if (finish_partials<RED_THREADS>(partial, out, arrived, 1, 0, m) && step.time != nullptr) {
#pragma clang fp contract(off)
        next_step(step, step.cfl * max_dt_of(step.N, m));
    }
}

// Block sums of per-thread values into partial[blockIdx.x * m + c0 + v].
template <int THREADS>
__device__ __forceinline__ void block_sums(double x, double* red, double* dst) {
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) x += __shfl_xor(x, w);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = red[0];
        for (int w = 1; w < THREADS / 64; ++w) s += red[w];
        store_partial(dst, s);
    }
    __syncthreads();
}

// sum_e J_e^d sum_n w_n u: each group of 16 lanes its nodes of 16 elements.
template <int DIM, int N>
__global__ void __launch_bounds__(RED_THREADS) integrate_kernel(const double* __restrict__ u,
                                                                const double* __restrict__ invJ,
                                                                double* __restrict__ partial, double* out,
                                                                unsigned* arrived, const double* __restrict__ w_g,
                                                                int64_t E, int nv) {
    constexpr int nn = cpow(N, DIM);
    __shared__ double red[RED_THREADS / 64];
    const int c = threadIdx.x % RED_ELEMS, g = threadIdx.x / RED_ELEMS;
    double acc[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) acc[v] = 0.0;
    for (int64_t e0 = (int64_t)blockIdx.x * RED_ELEMS; e0 < E; e0 += (int64_t)gridDim.x * RED_ELEMS) {
        const int64_t e = e0 + c;
        if (e >= E) continue;
        const double h = 1.0 / invJ[e];
        double vj = h;
#pragma unroll
        for (int d = 1; d < DIM; ++d) vj *= h;
#pragma unroll 4
        for (int n = g; n < nn; n += RED_GROUPS) {
            double w = vj;
            int r = n;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                w *= w_g[r % N];
                r /= N;
            }
#pragma unroll
            for (int v = 0; v < 9; ++v)
                if (v < nv) acc[v] += w * u[((int64_t)v * nn + n) * E + e];
        }
    }
#pragma unroll
    for (int v = 0; v < 9; ++v)
        if (v < nv) block_sums<RED_THREADS>(acc[v], red, &partial[(int64_t)blockIdx.x * nv + v]);
    finish_partials<RED_THREADS>(partial, out, arrived, nv, nv);
}

// Error norms against an initial condition on the tensor grid of NA = 2N - 1
// Lobatto nodes per direction: one wave per element interpolates one direction
// after the other through LDS (nv (N NA N^(d-1) + N NA^2 N^(d-2) + ...)
// products instead of nv (N NA)^d), then each lane takes its analysis points.
// The node coordinates are products of per-direction ones (TreeMesh elements
// are cubes), so each is interpolated along its own direction.
template <int DIM, int N>
constexpr int en_wave_doubles(int nv) {
    constexpr int NA = 2 * N - 1;
    return nv * (DIM > 1 ? NA * cpow(N, DIM - 1) : 0) + nv * (DIM > 2 ? NA * NA * N : 0) + DIM * NA;
}
// EXACT: the state compared against.  The waves of the convergence tests, which
// error norms are mostly taken against, have kernels of their own; the others
// go through the general function, a call per point with its registers and stack
// (82 us against 48 at 4096 elements of 3D Euler).
constexpr int EN_GENERAL = 0, EN_EULER_WAVE = 1, EN_ADVECTION_WAVE = 2;
template <int DIM, int N, int EXACT>
__global__ void __launch_bounds__(256) error_norms_kernel(const double* __restrict__ u, const double* __restrict__ xs,
                                                          const double* __restrict__ invJ,
                                                          double* __restrict__ partial, double* out,
                                                          unsigned* arrived, const double* __restrict__ Vdm_g,
                                                          const double* __restrict__ wa_g, int64_t E, IcParams q,
                                                          double t, int nv_) {
    const int nv = EXACT == EN_EULER_WAVE ? DIM + 2 : (EXACT == EN_ADVECTION_WAVE ? 1 : nv_);
    constexpr int NA = 2 * N - 1, NL = cpow(N, DIM - 1), NN = cpow(N, DIM), NP = cpow(NA, DIM);
    extern __shared__ double dyn[];
    __shared__ double V[NA * N], wa[NA], red[4][18];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, waves = blockDim.x / 64;
    for (int i = threadIdx.x; i < NA * N; i += blockDim.x) V[i] = Vdm_g[i];
    for (int i = threadIdx.x; i < NA; i += blockDim.x) wa[i] = wa_g[i];
    double* const xa = dyn + (int64_t)wave * en_wave_doubles<DIM, N>(nv);
    double* const s1 = xa + DIM * NA;                              // [v][a0][line]
    double* const s2 = s1 + (DIM > 1 ? nv * NA * NL : 0);          // [v][a0][a1][k]
    double l2[9], li[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) l2[v] = li[v] = 0.0;
    __syncthreads();
    for (int64_t base = (int64_t)blockIdx.x * waves; base < E; base += (int64_t)gridDim.x * waves) {
        const bool valid = base + wave < E;
        const int64_t e = valid ? base + wave : E - 1;
        for (int i = lane; i < DIM * NA; i += 64) {
            const int d = i / NA, a = i % NA;
            double x = 0.0;
#pragma unroll
            for (int p = 0; p < N; ++p) x += V[a * N + p] * xs[((int64_t)d * NN + p * cpow(N, d)) * E + e];
            xa[i] = x;
        }
        if constexpr (DIM > 1) {
            for (int i = lane; i < nv * NL; i += 64) {
                const int v = i / NL, l = i % NL;
                double val[N];
#pragma unroll
                for (int p = 0; p < N; ++p) val[p] = u[((int64_t)v * NN + l * N + p) * E + e];
#pragma unroll
                for (int a = 0; a < NA; ++a) {
                    double x = 0.0;
#pragma unroll
                    for (int p = 0; p < N; ++p) x += V[a * N + p] * val[p];
                    s1[(v * NA + a) * NL + l] = x;
                }
            }
        }
        __syncthreads();
        if constexpr (DIM > 2) {
            for (int i = lane; i < nv * NA * N; i += 64) {
                const int va = i / N, k = i % N;
                double val[N];
#pragma unroll
                for (int p = 0; p < N; ++p) val[p] = s1[va * NL + k * N + p];
#pragma unroll
                for (int a = 0; a < NA; ++a) {
                    double x = 0.0;
#pragma unroll
                    for (int p = 0; p < N; ++p) x += V[a * N + p] * val[p];
                    s2[(va * NA + a) * N + k] = x;
                }
            }
            __syncthreads();
        }
        const double h = 1.0 / invJ[e];
        double vj = h;
#pragma unroll
        for (int d = 1; d < DIM; ++d) vj *= h;
        for (int p = lane; p < NP && valid; p += 64) {
            int ai[3] = {0, 0, 0}, r = p;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                ai[d] = r % NA;
                r /= NA;
            }
            double x[3] = {0.0, 0.0, 0.0}, wq = vj;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                x[d] = xa[d * NA + ai[d]];
                wq *= wa[ai[d]];
            }
            double uex[9];
            if constexpr (EXACT == EN_EULER_WAVE) {
                double xs = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) xs += x[d];
                const double ini = euler_wave(xs, t);
#pragma unroll
                for (int v = 0; v < 9; ++v) uex[v] = v == DIM + 1 ? ini * ini : ini;
            } else if constexpr (EXACT == EN_ADVECTION_WAVE) {
                double xs = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) xs += x[d] - q.a[d] * t;
                const double w = advection_wave(xs);
#pragma unroll
                for (int v = 0; v < 9; ++v) uex[v] = w;
            } else {
                double ug[9];
                initial_condition(q, x, t, 0, ug);
#pragma unroll
                for (int v = 0; v < 9; ++v) uex[v] = v < nv ? ug[v] : 0.0;
            }
            const double* Vl = V + ai[DIM - 1] * N;
#pragma unroll
            for (int v = 0; v < 9; ++v) {
                if (v >= nv) continue;
                double ua = 0.0;
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    double f;
                    if constexpr (DIM == 1)
                        f = u[((int64_t)v * NN + j) * E + e];
                    else if constexpr (DIM == 2)
                        f = s1[(v * NA + ai[0]) * NL + j];
                    else
                        f = s2[((v * NA + ai[0]) * NA + ai[1]) * N + j];
                    ua += Vl[j] * f;
                }
                const double diff = uex[v] - ua;
                l2[v] += diff * diff * wq;
                li[v] = fmax(li[v], fabs(diff));
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < 9; ++v) {
        double a = l2[v], b = li[v];
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) {
            a += __shfl_xor(a, w);
            b = fmax(b, __shfl_xor(b, w));
        }
        if (lane == 0) {
            red[wave][v] = a;
            red[wave][9 + v] = b;
        }
    }
    __syncthreads();
    if (threadIdx.x < 9 && (int)threadIdx.x < nv) {
        const int v = threadIdx.x;
        double a = red[0][v], b = red[0][9 + v];
        for (int w = 1; w < waves; ++w) {
            a += red[w][v];
            b = fmax(b, red[w][9 + v]);
        }
        store_partial(&partial[(int64_t)blockIdx.x * 2 * nv + v], a);
        store_partial(&partial[(int64_t)blockIdx.x * 2 * nv + nv + v], b);
    }
    // (the last block's waves: as many as this block has)
    if (blockDim.x == 256)
        finish_partials<256>(partial, out, arrived, 2 * nv, nv);
    else if (blockDim.x == 128)
        finish_partials<128>(partial, out, arrived, 2 * nv, nv);
    else
        finish_partials<64>(partial, out, arrived, 2 * nv, nv);
}

}  // namespace trixi_hip
