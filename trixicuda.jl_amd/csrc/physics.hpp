// physics.hpp -- device-side equations and numerical fluxes for the gfx950
// DGSEM kernels.  Everything is templated on the arithmetic type R (double in
// the FP64 mode, float in the mixed modes) and on the type L of the per-node
// logarithms inside the entropy-conservative means (double in the FP64 and
// mixed modes; float only in the mixed_f32log mode, where the closed-form
// ln-mean, taken where |log y - log x| > 0.02, carries up to about 5e-6
// relative error from FP32 logarithms).
//
// The flux algebra follows the Trixi.jl definitions that TrixiCUDA.jl's
// kernels inline (reference: fluxes passed in by the tests, e.g.
// test/tree_dgsem_3d/euler_ec.jl:13-17, test/tree_dgsem_3d/mhd_alfven_wave.jl:13-18;
// call sites dg_3d_kernel.jl:221-234, 1155-1203).  Orientation o is 0-based.
//
// Node data.  Each equation defines a Node (primitive variables plus, where
// an entropy-conservative flux needs them, log(rho) and log(p)) built once
// per node from the conservative state; the conservative variables are
// reconstructed on demand (Node::cons) where a flux needs them.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "fastlog.hpp"

namespace trixi_hip {

// b^e; a loop rather than recursion, so that a call with a runtime exponent
// inlines instead of becoming a recursive device call (with a dynamic stack)
__host__ __device__ constexpr int cpow(int b, int e) {
    int r = 1;
    for (int i = 0; i < e; ++i) r *= b;
    return r;
}

enum Equation : int {
    EQ_LINADV = 0,
    EQ_EULER = 1,
    EQ_GLM_MHD = 2,
    EQ_BURGERS = 3,
    EQ_HYPDIFF = 4,
    EQ_EULER_MULTI = 5,
    EQ_EULER_QUASI1D = 6,
    EQ_SHALLOW_WATER = 7
};
constexpr int MAXC = 4;  // gas components of multicomponent Euler (parameter slots)
enum VolumeIntegral : int { VI_WEAK = 0, VI_FD = 1, VI_HG = 2 };
enum Flux : int {
    FLUX_CENTRAL = 0,
    FLUX_LLF = 1,         // FluxLaxFriedrichs(max_abs_speed)
    FLUX_LLF_NAIVE = 2,   // FluxLaxFriedrichs(max_abs_speed_naive)
    FLUX_RANOCHA = 3,
    FLUX_SHIMA_ETAL = 4,
    FLUX_HINDENLANG_GASSNER = 5,
    FLUX_EC = 6,          // flux_ec of the inviscid Burgers equation
    FLUX_HLL = 7,         // FluxHLL(min_max_speed_davis) (compressible Euler)
    FLUX_CHAN_ETAL = 8,   // flux_chan_etal + flux_nonconservative_chan_etal (quasi-1D Euler)
    FLUX_HLLE = 9,        // flux_hlle = FluxHLL(min_max_speed_einfeldt) (GLM-MHD)
    FLUX_WINTERMEYER_ETAL = 10,  // shallow water (volume; nonconservative term g h_l b_r)
    FLUX_FJORDHOLM_ETAL = 11,    // shallow water (surface; nonconservative term g h_l b_l + g h_avg [[b]])
    FLUX_HYDROSTATIC_LLF = 12    // shallow water: LLF of Audusse's hydrostatic reconstruction (+ Audusse's term)
};

// two-point fluxes that take ln-means (they need log(rho), log(p) per node)
constexpr bool flux_needs_logs(int f) {
    return f == FLUX_RANOCHA || f == FLUX_HINDENLANG_GASSNER || f == FLUX_CHAN_ETAL;
}

struct PhysParams {
    double gamma, inv_gm1, gm1, c_h;
    double a[3];
    double nu, inv_Tr;  // hyperbolic diffusion: diffusion constant, 1 / reference time
    // multicomponent Euler: per component c_v = R / (gamma - 1) and c_v gamma
    double cv[MAXC], cvg[MAXC];
    double grav;  // shallow water: gravitational acceleration
};

template <typename R>
struct PhysR {
    R gamma, inv_gm1, gm1, c_h, a[3], nu, inv_Tr, cv[MAXC], cvg[MAXC], grav;
    __host__ __device__ static PhysR from(const PhysParams& p) {
        PhysR r;
        r.gamma = (R)p.gamma;
        r.inv_gm1 = (R)p.inv_gm1;
        r.gm1 = (R)p.gm1;
        r.c_h = (R)p.c_h;
        r.nu = (R)p.nu;
        r.inv_Tr = (R)p.inv_Tr;
        r.grav = (R)p.grav;
        for (int d = 0; d < 3; ++d) r.a[d] = (R)p.a[d];
        for (int k = 0; k < MAXC; ++k) {
            r.cv[k] = (R)p.cv[k];
            r.cvg[k] = (R)p.cvg[k];
        }
        return r;
    }
};

// Index (v*NN + node)*E + e of an element-innermost state array: the
// uniform v*NN*E (`slab` = NN*E) stays in scalar registers and node*E + e is
// one 32x32->64-bit multiply-add per lane.  Exact for node, e >= 0 and
// E < 2^31 (element ids are int32).
__device__ __forceinline__ int64_t soa(int v, int node, int64_t e, int64_t slab, uint32_t E32) {
    return (int64_t)v * slab + (int64_t)((uint64_t)(uint32_t)node * (uint64_t)E32 + (uint64_t)e);
}

// ---------------------------------------------------------------------------
// arithmetic helpers.
//   FP64: reciprocal = v_rcp_f64 (relative error below 2^-24, measured)
//         refined by one third-order step r (1 + e + e^2), e = 1 - d r (the
//         remaining e^3 is below 2^-72), quotient n * r corrected by one
//         residual step (within about 1 ulp, far inside the FP64 parity
//         bound, 6 instructions instead of the 11-instruction IEEE sequence);
//         square root = v_rsq_f64 with one coupled (Goldschmidt) step and one
//         residual correction (measured over 2^18 arguments per range: correctly
//         rounded from 2^-1000 up, within 1 ulp down to the smallest normal
//         number, relative error 4e-15 of subnormal ones, whose residual is lost;
//         0 and infinity as they are).
//   FP32 (mixed mode): v_rcp_f32 and v_sqrt_f32 (within 2 ulp of FP32).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double rrcp(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, r, 1.0);
    return fma(r, fma(e, e, e), r);
}
__device__ __forceinline__ float rrcp(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double rdiv(double n, double d) {
    const double r = rrcp(d);
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}
__device__ __forceinline__ float rdiv(float n, float d) { return n * __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double rsqrt_(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;  // 0x260: -0, +0, +inf
}
__device__ __forceinline__ float rsqrt_(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double dabs(double x) { return fabs(x); }
__device__ __forceinline__ float dabs(float x) { return fabsf(x); }
template <typename R> __device__ __forceinline__ R dmax(R a, R b) { return b > a ? b : a; }

// Logarithms of the node records: fast_log in FP64 (about half the
// instructions of the library's log, within 2 ulp), the library's FP32 log
// in FP32.
__device__ __forceinline__ double node_log(double x) { return fast_log(x); }
__device__ __forceinline__ float node_log(float x) { return logf(x); }

// ---------------------------------------------------------------------------
// Logarithmic means (Trixi.jl ln_mean / inv_ln_mean) from per-node
// logarithms, branch free with a single reciprocal each.
//   f2 = ((y - x) / (x + y))^2; the series branch is taken for f2 < 1e-4,
//   tested as |y - x| < 0.01 (x + y) (x, y > 0; one product, the absolute
//   value is a source modifier; both branches are accurate to round-off on
//   either side of the threshold, so its exact placement does not matter).
//   series:  ln_mean     = (x + y) Q(f2),  Q = 1/P expanded to the order of
//                          P(f2) = 2 + 2f2/3 + 2f2^2/5 + 2f2^3/7:
//                          Q = 1/2 - f2/6 - 2 f2^2/45 - 22 f2^3/945
//                          (differs from 1/P by O(f2^4) < 1e-16 relative);
//            inv_ln_mean = P(f2) / (x + y);
//   closed:  ln_mean     = (y - x) / (log y - log x), inv_ln_mean = 1 / that.
//   The one reciprocal is of (x + y) in the series branch and of the
//   closed-branch denominator otherwise.  The logarithms and their
//   difference are in L: |log(y/x)| > 0.02 in the closed branch, so the
//   difference is accurate to a few 1e-14 with FP64 logarithms (then rounded
//   once to R) and to a few 1e-6 with FP32 ones.
// ---------------------------------------------------------------------------
template <typename R, typename L>
__device__ __forceinline__ R ln_mean_logs(R x, R y, L lx, L ly) {
    const R dxy = y - x, s = x + y;
    const bool series = dabs(dxy) < R(0.01) * s;
    const R r = rrcp(series ? s : (R)(ly - lx));
    const R z = dxy * r, f2 = z * z;
    const R q = R(0.5) + f2 * (R(-1.0 / 6.0) + f2 * (R(-2.0 / 45.0) + f2 * R(-22.0 / 945.0)));
    return series ? s * q : z;
}

template <typename R, typename L>
__device__ __forceinline__ R inv_ln_mean_logs(R x, R y, L lx, L ly) {
    const R dxy = y - x, s = x + y;
    const bool series = dabs(dxy) < R(0.01) * s;
    const R dl = (R)(ly - lx);
    const R r = rrcp(series ? s : dxy);
    const R z = dxy * r, f2 = z * z;
    const R pp = R(2) + f2 * (R(2.0 / 3.0) + f2 * (R(2.0 / 5.0) + f2 * R(2.0 / 7.0)));
    return series ? pp * r : dl * r;
}

// ---------------------------------------------------------------------------
// The two logarithmic means of an entropy-conservative flux without node
// logarithms (FP64 arithmetic): ln_mean(x1, y1) and inv_ln_mean(x2, y2) from
// the series in z^2, z = (y - x) / (x + y).
//   log(y / x) = z P(z^2), P(q) = 2 atanh(sqrt q) / sqrt q, and Q = 1 / P:
//   minimax polynomials of degree 6 for |z| < 0.15 (y / x < 1.353), relative
//   error of the stored coefficients below 5.2e-17 (P) and 1.1e-17 (Q), less than
//   half a unit in the last place.
// MEANS_NEAR: the caller knows that |z| < 0.15 for both (near_line).  MEANS_ANY:
// any x, y; lanes further apart take the closed form with the logarithm of the
// quotient, in a block that a wave without such lanes skips.
// Against node logarithms (two per node, staged in LDS) with a three-term
// series below |z| = 0.01, the FP64 kernels drop the logarithms, their LDS and
// registers, and every select and branch of a pair.
// ---------------------------------------------------------------------------
// MEANS_LOGS: from the nodes' logarithms after all.
constexpr int MEANS_LOGS = 0, MEANS_NEAR = 1, MEANS_ANY = 2;

// v_min_f64 / v_max_f64 as they are (fmin and fmax first quiet each operand
// with an instruction of its own); a NaN operand yields the other one
__device__ __forceinline__ double raw_min(double x, double y) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
__device__ __forceinline__ double raw_max(double x, double y) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
// y / x < 1.15 / 0.85 for x <= y (false for x <= 0 and for NaN)
__device__ __forceinline__ bool near_ratio(double x, double y) { return 0.85 * y < 1.15 * x; }

// 1 / s1 and 1 / s2 of the sums of two means, MEANS_NEAR from one reciprocal of
// their product (rho^2 p in size, which near_range keeps inside the FP64 range; two
// reciprocals take 0.5 us more of 80 in 3D at 32768 elements and 0.3 of 22 in 2D).
template <int MEANS>
__device__ __forceinline__ void sum_reciprocals(double s1, double s2, double& r1, double& r2) {
    if constexpr (MEANS == MEANS_NEAR) {
        const double r = rrcp(s1 * s2);
        r1 = r * s2;
        r2 = r * s1;
    } else {
        r1 = rrcp(s1);
        r2 = rrcp(s2);
    }
}
// whether the products s1 s2 of a line whose ratios are near lie well inside the
// FP64 range, by one of its nodes (the others' within a factor of 20)
__device__ __forceinline__ bool near_range(double rho, double p) {
    const double w = rho * (rho * p);
    return w > 0x1p-960 && w < 0x1p960;
}

template <int MEANS>
__device__ __forceinline__ void log_free_means(double x1, double y1, double x2, double y2, double& mean1,
                                               double& inv_mean2) {
    const double s1 = x1 + y1, d1 = y1 - x1;
    const double s2 = x2 + y2, d2 = y2 - x2;
    double r1, r2;
    sum_reciprocals<MEANS>(s1, s2, r1, r2);
    const double z1 = d1 * r1, z2 = d2 * r2;
    const double q1 = z1 * z1, q2 = z2 * z2;
    double Q = fma(q1, fastlog_const<true>(-0.008948152998574805), fastlog_const<true>(-0.01088099532782093));
    Q = fma(q1, Q, fastlog_const<true>(-0.015097271029888403));
    Q = fma(q1, Q, fastlog_const<true>(-0.023280421147242054));
    Q = fma(q1, Q, fastlog_const<true>(-0.0444444444524844));
    Q = fma(q1, Q, fastlog_const<true>(-0.1666666666666553));
    Q = fma(q1, Q, 0.5);
    double Pq = fma(q2, fastlog_const<true>(0.16481117002486795), fastlog_const<true>(0.1814740093132822));
    Pq = fma(q2, Pq, fastlog_const<true>(0.2222275413776025));
    Pq = fma(q2, Pq, fastlog_const<true>(0.28571424363123693));
    Pq = fma(q2, Pq, fastlog_const<true>(0.4000000001583343));
    Pq = fma(q2, Pq, fastlog_const<true>(0.6666666666664435));
    Pq = fma(q2, Pq, 2.0);
    mean1 = s1 * Q;
    inv_mean2 = Pq * r2;
    if constexpr (MEANS == MEANS_ANY) {
        // (false for nonpositive sums and NaN, which then go through the logarithm)
        const bool near1 = fabs(d1) < 0.15 * s1, near2 = fabs(d2) < 0.15 * s2;
        if (__builtin_amdgcn_ballot_w64(!(near1 && near2)) != 0) {
            const double nan = __builtin_nan("");
            const double l1 = x1 > 0.0 ? fast_log<true>(rdiv(y1, x1)) : nan;
            const double l2 = x2 > 0.0 ? fast_log<true>(rdiv(y2, x2)) : nan;
            mean1 = near1 ? mean1 : rdiv(d1, l1);
            inv_mean2 = near2 ? inv_mean2 : rdiv(l2, d2);
        }
    }
}

// ===========================================================================
// Linear scalar advection in DIM dimensions: u_t + a . grad u = 0.
// ===========================================================================
template <int DIM>
struct LinAdv {
    static constexpr int NV = 1;
    static constexpr bool NONCONS = false;
    static constexpr int NRF = 1;  // node record: u
    template <typename R, typename L = R>
    struct Node {
        R u;
        L lrho, lp;  // unused
        __device__ R cons(int) const { return u; }
    };
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>&) {
        Node<R, L> n;
        n.u = u[0];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        f[0] = n.u;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L, L, const PhysR<R>&) {
        Node<R, L> n;
        n.u = f[0];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
        f[0] = P.a[o] * n.u;
    }
    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        const R fl = P.a[o] * l.u, fr = P.a[o] * r.u;
        if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
            const R lam = dabs(P.a[o]);
            f[0] = R(0.5) * (fl + fr) + (R(-0.5) * lam * (r.u - l.u));
        } else {
            f[0] = R(0.5) * (fl + fr);
        }
    }
    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        for (int d = 0; d < DIM; ++d) lam[d] = dabs(P.a[d]);
    }
};

// ===========================================================================
// Hyperbolic diffusion (Trixi HyperbolicDiffusionEquations{1,2,3}D): (phi,
// q_1..DIM), the first-order hyperbolic system phi_t - nu div q = f,
// q_t - (grad phi - q) / T_r = 0 whose steady state solves -nu lap phi = f.
// Flux in direction o: f_phi = -nu q_o, f_{q_o} = -phi / T_r, others 0; the
// wave speed of LLF is the constant sqrt(nu / T_r).
// ===========================================================================
template <int DIM>
struct HypDiff {
    static constexpr int NV = DIM + 1;
    static constexpr bool NONCONS = false;
    static constexpr int NRF = DIM + 1;
    template <typename R, typename L = R>
    struct Node {
        R u[DIM + 1];
        L lrho, lp;  // unused
        __device__ R cons(int q) const { return u[q]; }
    };
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>&) {
        Node<R, L> n;
#pragma unroll
        for (int q = 0; q < NV; ++q) n.u[q] = u[q];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
#pragma unroll
        for (int q = 0; q < NV; ++q) f[q] = n.u[q];
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L, L, const PhysR<R>&) {
        Node<R, L> n;
#pragma unroll
        for (int q = 0; q < NV; ++q) n.u[q] = f[q];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
        f[0] = -P.nu * n.u[1 + o];
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = (d == o) ? -n.u[0] * P.inv_Tr : R(0);
    }
    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        R fl[NV], fr[NV];
        flux(l, o, P, fl);
        flux(r, o, P, fr);
        if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
            const R lam = sqrt(P.nu * P.inv_Tr);
#pragma unroll
            for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]) + (R(-0.5) * lam * (r.u[q] - l.u[q]));
        } else {
#pragma unroll
            for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]);
        }
    }
    template <typename R>
    __device__ static void max_abs_speeds(const R*, const PhysR<R>& P, R* lam) {
#pragma unroll
        for (int d = 0; d < DIM; ++d) lam[d] = sqrt(P.nu * P.inv_Tr);
    }
};

// ===========================================================================
// Inviscid Burgers equation in 1D (Trixi InviscidBurgersEquation1D):
// u_t + (u^2 / 2)_x = 0.  flux_ec is the entropy-conservative two-point flux
// (u_l^2 + u_l u_r + u_r^2) / 6 for the entropy u^2 / 2; the wave speed of
// both LLF variants is max(|u_l|, |u_r|).
// ===========================================================================
struct Burgers {
    static constexpr int NV = 1;
    static constexpr bool NONCONS = false;
    static constexpr int NRF = 1;
    template <typename R, typename L = R>
    struct Node {
        R u;
        L lrho, lp;  // unused
        __device__ R cons(int) const { return u; }
    };
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>&) {
        Node<R, L> n;
        n.u = u[0];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        f[0] = n.u;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L, L, const PhysR<R>&) {
        Node<R, L> n;
        n.u = f[0];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int, const PhysR<R>&, R* f) {
        f[0] = R(0.5) * n.u * n.u;
    }
    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int, const PhysR<R>&, R* f) {
        if (KIND == FLUX_EC) {
            f[0] = (l.u * l.u + l.u * r.u + r.u * r.u) * R(1.0 / 6.0);
        } else {
            const R fl = R(0.5) * l.u * l.u, fr = R(0.5) * r.u * r.u;
            if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
                const R lam = dmax(dabs(l.u), dabs(r.u));
                f[0] = R(0.5) * (fl + fr) + (R(-0.5) * lam * (r.u - l.u));
            } else {
                f[0] = R(0.5) * (fl + fr);
            }
        }
    }
    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>&, R* lam) {
        lam[0] = dabs(u[0]);
    }
};

// ===========================================================================
// Compressible Euler in DIM dimensions: (rho, rho v_1..DIM, rho e).
// ===========================================================================
template <int DIM>
struct Euler {
    static constexpr int NV = DIM + 2;
    static constexpr bool NONCONS = false;
    static constexpr int NRF = DIM + 3;  // node record: rho, v[DIM], p, c
    template <typename R, typename L = R>
    struct Node {
        R rho, v[DIM], p, c;  // primitives and sound speed
        L lrho, lp;      // log(rho), log(p) for the entropy-conservative means
        R inv_gm1;
        __device__ R cons(int q) const {
            if (q == 0) return rho;
            if (q <= DIM) return rho * v[q - 1];
            R ke = R(0);
#pragma unroll
            for (int d = 0; d < DIM; ++d) ke += rho * v[d] * v[d];
            return p * inv_gm1 + R(0.5) * ke;
        }
    };

    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>& P) {
        Node<R, L> n;
        n.rho = u[0];
        const R inv_rho = rdiv(R(1), n.rho);
        R ke = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            n.v[d] = u[1 + d] * inv_rho;
            ke = (d == 0) ? u[1 + d] * n.v[d] : ke + u[1 + d] * n.v[d];
        }
        n.p = P.gm1 * (u[DIM + 1] - R(0.5) * ke);
        n.c = rsqrt_(P.gamma * n.p * inv_rho);
        n.inv_gm1 = P.inv_gm1;
        if (LOGS) {
            n.lrho = node_log((L)n.rho);
            n.lp = node_log((L)n.p);
        } else {
            n.lrho = n.lp = 0.0;
        }
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        f[0] = n.rho;
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = n.v[d];
        f[DIM + 1] = n.p;
        f[DIM + 2] = n.c;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L lrho, L lp, const PhysR<R>& P) {
        Node<R, L> n;
        n.rho = f[0];
#pragma unroll
        for (int d = 0; d < DIM; ++d) n.v[d] = f[1 + d];
        n.p = f[DIM + 1];
        n.c = f[DIM + 2];
        n.lrho = lrho;
        n.lp = lp;
        n.inv_gm1 = P.inv_gm1;
        return n;
    }

    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
        const R rho_vo = n.rho * n.v[o];
        f[0] = rho_vo;
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = (d == o) ? rho_vo * n.v[d] + n.p : rho_vo * n.v[d];
        f[DIM + 1] = (n.cons(DIM + 1) + n.p) * n.v[o];
    }

    // flux_ranocha from its logarithmic means
    template <typename R, typename L>
    __device__ static void ranocha(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R rho_mean,
                                   R inv_rho_p_mean, R* f) {
        R vavg[DIM];
        R vsq = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            vavg[d] = R(0.5) * (l.v[d] + r.v[d]);
            vsq = (d == 0) ? l.v[d] * r.v[d] : vsq + l.v[d] * r.v[d];
        }
        const R velocity_square_avg = R(0.5) * vsq;
        const R p_avg = R(0.5) * (l.p + r.p);
        const R f1 = rho_mean * vavg[o];
        f[0] = f1;
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = (d == o) ? f1 * vavg[d] + p_avg : f1 * vavg[d];
        f[DIM + 1] = f1 * (velocity_square_avg + inv_rho_p_mean * P.inv_gm1) +
                     R(0.5) * (l.p * r.v[o] + r.p * l.v[o]);
    }

    // Twice a two-point flux (FP64): the factors 1/2 of the averages and of the
    // Lax-Friedrichs flux go into the kernel's final factor.
    // FLUX_RANOCHA without node logarithms: with V = v_l + v_r and h = ln_mean(rho) V_o / 2,
    //   2 f = (2 h, h V + (p_l + p_r) e_o,
    //          h (v_l . v_r + 2 / (gamma - 1) p_l p_r inv_ln_mean) + p_l v_r,o + p_r v_l,o).
    // FLUX_SHIMA_ETAL: the same with h = (rho_l + rho_r) V_o / 4 and the
    // energy's internal part (p_l + p_r) V_o / (2 (gamma - 1)).
    // FLUX_LLF*: with the conservative states u_l, u_r,
    //   2 f = v_l,o u_l + v_r,o u_r + lambda (u_l - u_r) + (0, (p_l + p_r) e_o, p_l v_l,o + p_r v_r,o).
    template <int KIND, int MEANS, typename L>
    __device__ static void twice_flux(const Node<double, L>& l, const double* ul, const Node<double, L>& r,
                                      const double* ur, int o, const PhysR<double>& P, double* f) {
        if constexpr (KIND == FLUX_SHIMA_ETAL) {
            const double Vo = l.v[o] + r.v[o], psum = l.p + r.p;
            f[0] = 0.5 * ((l.rho + r.rho) * Vo);
            const double h = 0.5 * f[0];
            double vsq = l.v[0] * r.v[0];
#pragma unroll
            for (int d = 1; d < DIM; ++d) vsq = fma(l.v[d], r.v[d], vsq);
#pragma unroll
            for (int d = 0; d < DIM; ++d) f[1 + d] = (d == o) ? fma(h, Vo, psum) : h * (l.v[d] + r.v[d]);
            const double e = fma(l.p, r.v[o], r.p * l.v[o]);
            f[DIM + 1] = fma(h, vsq, fma(0.5 * P.inv_gm1, psum * Vo, e));
        } else if constexpr (KIND == FLUX_RANOCHA) {
            double rho_mean, inv_mean;
            log_free_means<MEANS>(l.rho, r.rho, l.rho * r.p, r.rho * l.p, rho_mean, inv_mean);
            const double Vo = l.v[o] + r.v[o];
            f[0] = rho_mean * Vo;
            const double h = 0.5 * f[0];
            double vsq = l.v[0] * r.v[0];
#pragma unroll
            for (int d = 1; d < DIM; ++d) vsq = fma(l.v[d], r.v[d], vsq);
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                f[1 + d] = (d == o) ? fma(h, Vo, l.p + r.p) : h * (l.v[d] + r.v[d]);
            const double e = fma(l.p, r.v[o], r.p * l.v[o]);
            f[DIM + 1] = fma(h, fma(l.p * r.p * inv_mean, 2.0 * P.inv_gm1, vsq), e);
        } else {
            double lam;
            if (KIND == FLUX_LLF_NAIVE)
                lam = dmax(dabs(l.v[o]), dabs(r.v[o])) + dmax(l.c, r.c);
            else
                lam = dmax(dabs(l.v[o]) + l.c, dabs(r.v[o]) + r.c);
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                double t = fma(l.v[o], ul[q], r.v[o] * ur[q]);
                if (q == 1 + o) t += l.p + r.p;
                if (q == DIM + 1) t = fma(l.p, l.v[o], fma(r.p, r.v[o], t));
                f[q] = fma(lam, ul[q] - ur[q], t);
            }
        }
    }
    // whether every pair of these nodes satisfies MEANS_NEAR: rho, and rho / p
    // through the staged sound speed (rho / p = gamma / c^2).  Minimum and maximum
    // pass over a node that is not a number; the sum of the speeds does not, nor one
    // with p / rho < 0
    template <int N, class ND>
    __device__ static bool near_line(const ND* n) {
        double r0 = n[0].rho, r1 = r0, c0 = n[0].c, c1 = c0, sum = c0;
#pragma unroll
        for (int i = 1; i < N; ++i) {
            r0 = raw_min(r0, n[i].rho);
            r1 = raw_max(r1, n[i].rho);
            c0 = raw_min(c0, n[i].c);
            c1 = raw_max(c1, n[i].c);
            sum += n[i].c;
        }
        const bool a = near_ratio(r0, r1), b = near_ratio(c0 * c0, c1 * c1), c = sum < 0x1p1000;
        return a && b && c && near_range(n[0].rho, n[0].p);
    }

    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        if (KIND == FLUX_RANOCHA) {
            const R rho_mean = ln_mean_logs<R>(l.rho, r.rho, l.lrho, r.lrho);
            // p_ll p_rr inv_ln_mean(rho_ll p_rr, rho_rr p_ll), logs log(rho)+log(p)
            const R inv_rho_p_mean =
                l.p * r.p * inv_ln_mean_logs<R>(l.rho * r.p, r.rho * l.p, l.lrho + r.lp, r.lrho + l.lp);
            ranocha(l, r, o, P, rho_mean, inv_rho_p_mean, f);
        } else if (KIND == FLUX_SHIMA_ETAL) {
            const R rho_avg = R(0.5) * (l.rho + r.rho);
            R vavg[DIM];
            R ksum = R(0);
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                vavg[d] = R(0.5) * (l.v[d] + r.v[d]);
                ksum = (d == 0) ? l.v[d] * r.v[d] : ksum + l.v[d] * r.v[d];
            }
            const R kin_avg = R(0.5) * ksum;
            const R p_avg = R(0.5) * (l.p + r.p);
            const R pv_avg = R(0.5) * (l.p * r.v[o] + r.p * l.v[o]);
            const R f1 = rho_avg * vavg[o];
            f[0] = f1;
#pragma unroll
            for (int d = 0; d < DIM; ++d) f[1 + d] = (d == o) ? f1 * vavg[d] + p_avg : f1 * vavg[d];
            f[DIM + 1] = p_avg * vavg[o] * P.inv_gm1 + f1 * kin_avg + pv_avg;
        } else {
            R fl[NV], fr[NV];
            flux(l, o, P, fl);
            flux(r, o, P, fr);
            if (KIND == FLUX_HLL) {
                // HLL with Davis' estimates lambda_min = min(v_l - c_l, v_r - c_r),
                // lambda_max = max(v_l + c_l, v_r + c_r): upwind when both have
                // one sign, else (lmax f_l - lmin f_r + lmin lmax [[u]]) / (lmax - lmin)
                const R a = l.v[o] - l.c, b = r.v[o] - r.c, cc = l.v[o] + l.c, dd = r.v[o] + r.c;
                const R lmin = b < a ? b : a;
                const R lmax = dmax(cc, dd);
                if (lmin >= R(0) && lmax >= R(0)) {
#pragma unroll
                    for (int q = 0; q < NV; ++q) f[q] = fl[q];
                } else if (lmax <= R(0) && lmin <= R(0)) {
#pragma unroll
                    for (int q = 0; q < NV; ++q) f[q] = fr[q];
                } else {
                    const R inv = rdiv(R(1), lmax - lmin);
                    const R fll = lmax * inv, frr = lmin * inv, fdiss = lmin * lmax * inv;
#pragma unroll
                    for (int q = 0; q < NV; ++q) f[q] = fll * fl[q] - frr * fr[q] + fdiss * (r.cons(q) - l.cons(q));
                }
            } else if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
                R lam;
                if (KIND == FLUX_LLF_NAIVE)
                    lam = dmax(dabs(l.v[o]), dabs(r.v[o])) + dmax(l.c, r.c);
                else
                    lam = dmax(dabs(l.v[o]) + l.c, dabs(r.v[o]) + r.c);
                const R hl = R(-0.5) * lam;
#pragma unroll
                for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]) + hl * (r.cons(q) - l.cons(q));
            } else {
#pragma unroll
                for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]);
            }
        }
    }

    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        const R rho = u[0];
        R v[DIM], ke = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            v[d] = u[1 + d] / rho;
            ke = (d == 0) ? u[1 + d] * v[d] : ke + u[1 + d] * v[d];
        }
        const R p = P.gm1 * (u[DIM + 1] - R(0.5) * ke);
        const R c = sqrt(P.gamma * p / rho);
#pragma unroll
        for (int d = 0; d < DIM; ++d) lam[d] = dabs(v[d]) + c;
    }

    // density * pressure (Trixi density_pressure), the HG indicator variable
    template <typename R>
    __device__ static R density_pressure(const R* u, const PhysR<R>& P) {
        R ke = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) ke = (d == 0) ? u[1 + d] * u[1 + d] : ke + u[1 + d] * u[1 + d];
        return P.gm1 * (u[0] * u[DIM + 1] - R(0.5) * ke);
    }

    // the HG indicator variable: 0 density * pressure, 1 pressure (Trixi
    // pressure), 2 density
    __device__ static double indicator_variable(const double* u, const PhysR<double>& P, int var) {
        if (var == 2) return u[0];
        if (var == 1) {
            double ke = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) ke += u[1 + d] * u[1 + d];
            return P.gm1 * (u[DIM + 1] - 0.5 * ke / u[0]);
        }
        return density_pressure(u, P);
    }
};

// ===========================================================================
// Multicomponent compressible Euler (Trixi CompressibleEulerMulticomponent-
// Equations{1,2}D): (rho v_1..DIM, rho e, rho_1..rho_NC).  The mixture has
// rho = sum rho_k and gamma = sum rho_k c_v,k gamma_k / sum rho_k c_v,k
// (Trixi totalgamma), p = (gamma - 1)(rho e - rho |v|^2 / 2).
// flux_ranocha is Trixi's multicomponent form: ln-means of the partial
// densities, the Euler momentum and energy structure with the gamma of the
// averaged state; the partial-density logarithms are taken per pair (the
// node record stages log(rho) and log(p) only).
// ===========================================================================
template <int DIM, int NC>
struct EulerMulti {
    static constexpr int NV = DIM + 1 + NC;
    static constexpr bool NONCONS = false;
    static constexpr int NRF = NC + DIM + 2;  // node record: rho_k[NC], v[DIM], p, c
    template <typename R, typename L = R>
    struct Node {
        R rk[NC], v[DIM], p, c;
        R rho, inv_gm1;   // derived: total density, 1 / (gamma - 1)
        L lrho, lp;  // log(rho), log(p)
        __device__ R cons(int q) const {
            if (q < DIM) return rho * v[q];
            if (q == DIM) {
                R ke = R(0);
#pragma unroll
                for (int d = 0; d < DIM; ++d) ke += rho * v[d] * v[d];
                return p * inv_gm1 + R(0.5) * ke;
            }
            return rk[q - DIM - 1];
        }
    };

    // sum rho_k c_v,k gamma_k and sum rho_k c_v,k
    template <typename R>
    __device__ static R gamma_of(const R* rk, const PhysR<R>& P) {
        R h1 = R(0), h2 = R(0);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            h1 += rk[k] * P.cvg[k];
            h2 += rk[k] * P.cv[k];
        }
        return rdiv(h1, h2);
    }

    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>& P) {
        Node<R, L> n;
        R rho = R(0);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            n.rk[k] = u[DIM + 1 + k];
            rho += n.rk[k];
        }
        n.rho = rho;
        const R inv_rho = rdiv(R(1), rho);
        R vsq = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            n.v[d] = u[d] * inv_rho;
            vsq += n.v[d] * n.v[d];
        }
        const R gamma = gamma_of(n.rk, P);
        n.p = (gamma - R(1)) * (u[DIM] - R(0.5) * rho * vsq);
        n.c = rsqrt_(gamma * n.p * inv_rho);
        n.inv_gm1 = rdiv(R(1), gamma - R(1));
        if (LOGS) {
            n.lrho = node_log((L)n.rho);
            n.lp = node_log((L)n.p);
        } else {
            n.lrho = n.lp = 0.0;
        }
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
#pragma unroll
        for (int k = 0; k < NC; ++k) f[k] = n.rk[k];
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[NC + d] = n.v[d];
        f[NC + DIM] = n.p;
        f[NC + DIM + 1] = n.c;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L lrho, L lp, const PhysR<R>& P) {
        Node<R, L> n;
        R rho = R(0);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            n.rk[k] = f[k];
            rho += f[k];
        }
        n.rho = rho;
#pragma unroll
        for (int d = 0; d < DIM; ++d) n.v[d] = f[NC + d];
        n.p = f[NC + DIM];
        n.c = f[NC + DIM + 1];
        n.inv_gm1 = rdiv(R(1), gamma_of(n.rk, P) - R(1));
        n.lrho = lrho;
        n.lp = lp;
        return n;
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[d] = (d == o) ? n.rho * n.v[d] * n.v[o] + n.p : n.rho * n.v[d] * n.v[o];
        f[DIM] = (n.cons(DIM) + n.p) * n.v[o];
#pragma unroll
        for (int k = 0; k < NC; ++k) f[DIM + 1 + k] = n.rk[k] * n.v[o];
    }

    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        if (KIND == FLUX_RANOCHA) {
            R f_rho_sum = R(0), ravg[NC];
            const R vo_avg = R(0.5) * (l.v[o] + r.v[o]);
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                const R fk = ln_mean_logs<R>(l.rk[k], r.rk[k], node_log((L)l.rk[k]), node_log((L)r.rk[k])) * vo_avg;
                f[DIM + 1 + k] = fk;
                f_rho_sum += fk;
                ravg[k] = R(0.5) * (l.rk[k] + r.rk[k]);
            }
            const R inv_gm1 = rdiv(R(1), gamma_of(ravg, P) - R(1));
            const R inv_rho_p_mean =
                l.p * r.p * inv_ln_mean_logs<R>(l.rho * r.p, r.rho * l.p, l.lrho + r.lp, r.lrho + l.lp);
            R vsq = R(0);
#pragma unroll
            for (int d = 0; d < DIM; ++d) vsq += l.v[d] * r.v[d];
            const R velocity_square_avg = R(0.5) * vsq;
            const R p_avg = R(0.5) * (l.p + r.p);
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const R vd = R(0.5) * (l.v[d] + r.v[d]);
                f[d] = (d == o) ? f_rho_sum * vd + p_avg : f_rho_sum * vd;
            }
            f[DIM] = f_rho_sum * (velocity_square_avg + inv_rho_p_mean * inv_gm1) +
                     R(0.5) * (l.p * r.v[o] + r.p * l.v[o]);
        } else {
            R fl[NV], fr[NV];
            flux(l, o, P, fl);
            flux(r, o, P, fr);
            if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
                R lam;
                if (KIND == FLUX_LLF_NAIVE)
                    lam = dmax(dabs(l.v[o]), dabs(r.v[o])) + dmax(l.c, r.c);
                else
                    lam = dmax(dabs(l.v[o]) + l.c, dabs(r.v[o]) + r.c);
                const R hl = R(-0.5) * lam;
#pragma unroll
                for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]) + hl * (r.cons(q) - l.cons(q));
            } else {
#pragma unroll
                for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]);
            }
        }
    }

    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        const Node<R> n = node<R, false>(u, P);
#pragma unroll
        for (int d = 0; d < DIM; ++d) lam[d] = dabs(n.v[d]) + n.c;
    }
};

// ===========================================================================
// Quasi-one-dimensional compressible Euler (Trixi
// CompressibleEulerEquationsQuasi1D): (a rho, a rho v, a e, a) with the nozzle
// width a, e = p / (gamma - 1) + rho v^2 / 2;
//   (a rho)_t + (a rho v)_x = 0,  (a rho v)_t + (a rho v^2)_x + a p_x = 0,
//   (a e)_t + (a v (e + p))_x = 0,  a_t = 0.
// flux_chan_etal is the entropy-conservative two-point flux of Chan et al.
// (2023) and flux_nonconservative_chan_etal(u_l, u_r) = (0, a_l p_r, 0, 0)
// the pressure-gradient term.
// ===========================================================================
struct EulerQuasi1D {
    static constexpr int NV = 4;
    static constexpr bool NONCONS = true;
    static constexpr int NRF = 5;  // node record: rho, v, p, c, a
    template <typename R, typename L = R>
    struct Node {
        R rho, v[1], p, c, a;
        L lrho, lp;
        R inv_gm1;
        __device__ R cons(int q) const {
            if (q == 0) return a * rho;
            if (q == 1) return a * rho * v[0];
            if (q == 2) return a * (p * inv_gm1 + R(0.5) * rho * v[0] * v[0]);
            return a;
        }
    };
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>& P) {
        Node<R, L> n;
        n.a = u[3];
        const R inv_a = rdiv(R(1), n.a);
        n.rho = u[0] * inv_a;
        const R rv = u[1] * inv_a;
        n.v[0] = rdiv(rv, n.rho);
        n.p = P.gm1 * (u[2] * inv_a - R(0.5) * rv * n.v[0]);
        n.c = rsqrt_(P.gamma * n.p * rdiv(R(1), n.rho));
        n.inv_gm1 = P.inv_gm1;
        if (LOGS) {
            n.lrho = node_log((L)n.rho);
            n.lp = node_log((L)n.p);
        } else {
            n.lrho = n.lp = 0.0;
        }
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        f[0] = n.rho;
        f[1] = n.v[0];
        f[2] = n.p;
        f[3] = n.c;
        f[4] = n.a;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L lrho, L lp, const PhysR<R>& P) {
        Node<R, L> n;
        n.rho = f[0];
        n.v[0] = f[1];
        n.p = f[2];
        n.c = f[3];
        n.a = f[4];
        n.lrho = lrho;
        n.lp = lp;
        n.inv_gm1 = P.inv_gm1;
        return n;
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int, const PhysR<R>& P, R* f) {
        const R arv = n.a * n.rho * n.v[0];
        f[0] = arv;
        f[1] = arv * n.v[0];
        f[2] = n.a * n.v[0] * (n.p * n.inv_gm1 + R(0.5) * n.rho * n.v[0] * n.v[0] + n.p);
        f[3] = R(0);
    }
    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        if (KIND == FLUX_CHAN_ETAL) {
            const R rho_mean = ln_mean_logs<R>(l.rho, r.rho, l.lrho, r.lrho);
            const R inv_rho_p_mean =
                l.p * r.p * inv_ln_mean_logs<R>(l.rho * r.p, r.rho * l.p, l.lrho + r.lp, r.lrho + l.lp);
            const R v_avg = R(0.5) * (l.v[0] + r.v[0]);
            const R a_v_avg = R(0.5) * (l.a * l.v[0] + r.a * r.v[0]);
            const R velocity_square_avg = R(0.5) * (l.v[0] * r.v[0]);
            const R f1 = rho_mean * a_v_avg;
            f[0] = f1;
            f[1] = f1 * v_avg;
            f[2] = f1 * (velocity_square_avg + inv_rho_p_mean * P.inv_gm1) +
                   R(0.5) * (l.p * r.a * r.v[0] + r.p * l.a * l.v[0]);
            f[3] = R(0);
        } else {
            R fl[NV], fr[NV];
            flux(l, o, P, fl);
            flux(r, o, P, fr);
            if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
                const R lam = dmax(dabs(l.v[0]), dabs(r.v[0])) + dmax(l.c, r.c);
#pragma unroll
                for (int q = 0; q < NV; ++q)
                    f[q] = R(0.5) * (fl[q] + fr[q]) + (R(-0.5) * lam * (r.cons(q) - l.cons(q)));
            } else {
#pragma unroll
                for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]);
            }
        }
    }
    template <int POS, typename R, typename L>
    __device__ static void noncons(const Node<R, L>& l, const Node<R, L>& r, int, const PhysR<R>&, R* f) {
        f[0] = R(0);
        f[1] = l.a * r.p;
        f[2] = R(0);
        f[3] = R(0);
    }
    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        const Node<R> n = node<R, false>(u, P);
        lam[0] = dabs(n.v[0]) + n.c;
    }
};

// ===========================================================================
// Shallow water (Trixi ShallowWaterEquations{1,2}D): (h, h v_1..DIM, b) with
// the bottom topography b; flux (h v_o, h v v_o + g h^2/2 e_o, 0) and the
// nonconservative bottom term g h grad b.  The volume pairs
// flux_wintermeyer_etal with g h_l b_r; at surfaces (and in shock-capturing
// subcells) the term belongs to the surface flux: Fjordholm's
// g h_l b_l + g (h_l + h_r)/2 (b_r - b_l), or, with the hydrostatic
// reconstruction, Audusse's g h_l b_l - g (h_l* + h_l)(h_l* - h_l) with
// h* = max(0, h + b - max(b_l, b_r)).  LLF does not dissipate b.
// ===========================================================================
template <int DIM>
struct ShallowWater {
    static constexpr int NV = DIM + 2;
    static constexpr bool NONCONS = true;
    static constexpr int NRF = DIM + 2;  // node record: h, v[DIM], b
    template <typename R, typename L = R>
    struct Node {
        R h, v[DIM], b;
        L lrho, lp;  // unused
        __device__ R cons(int q) const {
            if (q == 0) return h;
            if (q <= DIM) return h * v[q - 1];
            return b;
        }
    };
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>&) {
        Node<R, L> n;
        n.h = u[0];
        const R inv_h = rdiv(R(1), n.h);
#pragma unroll
        for (int d = 0; d < DIM; ++d) n.v[d] = u[1 + d] * inv_h;
        n.b = u[DIM + 1];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        f[0] = n.h;
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = n.v[d];
        f[DIM + 1] = n.b;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L, L, const PhysR<R>&) {
        Node<R, L> n;
        n.h = f[0];
#pragma unroll
        for (int d = 0; d < DIM; ++d) n.v[d] = f[1 + d];
        n.b = f[DIM + 1];
        n.lrho = n.lp = 0.0;
        return n;
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
        const R hvo = n.h * n.v[o];
        const R p = R(0.5) * P.grav * n.h * n.h;
        f[0] = hvo;
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = hvo * n.v[d] + (d == o ? p : R(0));
        f[DIM + 1] = R(0);
    }
    // LLF of two states, b not dissipated
    template <int KIND, typename R, typename L>
    __device__ static void llf(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        R fl[NV], fr[NV];
        flux(l, o, P, fl);
        flux(r, o, P, fr);
        const R cl = rsqrt_(P.grav * l.h), cr = rsqrt_(P.grav * r.h);
        R lam;
        if (KIND == FLUX_LLF_NAIVE)
            lam = dmax(dabs(l.v[o]), dabs(r.v[o])) + dmax(cl, cr);
        else
            lam = dmax(dabs(l.v[o]) + cl, dabs(r.v[o]) + cr);
        const R hl = R(-0.5) * lam;
#pragma unroll
        for (int q = 0; q <= DIM; ++q) f[q] = R(0.5) * (fl[q] + fr[q]) + hl * (r.cons(q) - l.cons(q));
        f[DIM + 1] = R(0);
    }
    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        if (KIND == FLUX_WINTERMEYER_ETAL || KIND == FLUX_FJORDHOLM_ETAL) {
            R f0, p_avg;
            if (KIND == FLUX_WINTERMEYER_ETAL) {
                f0 = R(0.5) * (l.h * l.v[o] + r.h * r.v[o]);
                p_avg = R(0.5) * P.grav * l.h * r.h;
            } else {
                f0 = R(0.5) * (l.h + r.h) * (R(0.5) * (l.v[o] + r.v[o]));
                p_avg = R(0.25) * P.grav * (l.h * l.h + r.h * r.h);
            }
            f[0] = f0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) f[1 + d] = f0 * (R(0.5) * (l.v[d] + r.v[d])) + (d == o ? p_avg : R(0));
            f[DIM + 1] = R(0);
        } else if (KIND == FLUX_HYDROSTATIC_LLF) {
            // FluxHydrostaticReconstruction(flux_lax_friedrichs,
            // hydrostatic_reconstruction_audusse_etal): LLF of the states with
            // h* = max(0, h + b - max(b_l, b_r)), the velocities kept
            const R bmax = dmax(l.b, r.b);
            Node<R, L> ls = l, rs = r;
            ls.h = dmax(R(0), l.h + l.b - bmax);
            rs.h = dmax(R(0), r.h + r.b - bmax);
            llf<FLUX_LLF>(ls, rs, o, P, f);
        } else if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
            llf<KIND>(l, r, o, P, f);
        } else {
            R fl[NV], fr[NV];
            flux(l, o, P, fl);
            flux(r, o, P, fr);
#pragma unroll
            for (int q = 0; q < NV; ++q) f[q] = R(0.5) * (fl[q] + fr[q]);
        }
    }
    // POS < 0: the volume term (flux_nonconservative_wintermeyer_etal); else
    // the term paired with surface / subcell flux POS
    template <int POS, typename R, typename L>
    __device__ static void noncons(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        R t;
        if (POS < 0) {
            t = P.grav * l.h * r.b;
        } else if (POS == FLUX_HYDROSTATIC_LLF) {
            const R hs = dmax(R(0), l.h + l.b - dmax(l.b, r.b));
            t = P.grav * l.h * l.b - P.grav * (hs + l.h) * (hs - l.h);
        } else {
            t = P.grav * l.h * l.b + P.grav * (R(0.5) * (l.h + r.h)) * (r.b - l.b);
        }
        f[0] = R(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) f[1 + d] = (d == o) ? t : R(0);
        f[DIM + 1] = R(0);
    }
    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        const Node<R> n = node<R, false>(u, P);
        const R c = rsqrt_(P.grav * n.h);
#pragma unroll
        for (int d = 0; d < DIM; ++d) lam[d] = dabs(n.v[d]) + c;
    }
    // waterheight_pressure = h g h^2 / 2, the HG indicator variable
    __device__ static double waterheight_pressure(const double* u, const PhysR<double>& P) {
        return u[0] * (0.5 * P.grav * u[0] * u[0]);
    }
};

// ===========================================================================
// Ideal GLM-MHD: (rho, rho v1..3, rho e, B1..3, psi), Powell and Galilean
// nonconservative terms.  IdealGlmMhdEquations3D uses orientations 0..2,
// IdealGlmMhdEquations2D the same nine-variable system with orientations 0, 1.
// ===========================================================================
struct GlmMhd {
    static constexpr int NV = 9;
    static constexpr bool NONCONS = true;
    static constexpr int NRF = 9;  // node record: rho, v[3], p, B[3], psi
    template <typename R, typename L = R>
    struct Node {
        R rho, v[3], p, B[3], psi;
        L lrho, lp;
        R inv_gm1;
        __device__ R cons(int q) const {
            if (q == 0) return rho;
            if (q <= 3) return rho * v[q - 1];
            if (q == 4)
                return p * inv_gm1 + R(0.5) * (rho * v[0] * v[0] + rho * v[1] * v[1] + rho * v[2] * v[2]) +
                       R(0.5) * (B[0] * B[0] + B[1] * B[1] + B[2] * B[2]) + R(0.5) * psi * psi;
            if (q <= 7) return B[q - 5];
            return psi;
        }
    };
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>& P) {
        Node<R, L> n;
        n.rho = u[0];
        const R inv_rho = rdiv(R(1), n.rho);
        n.v[0] = u[1] * inv_rho;
        n.v[1] = u[2] * inv_rho;
        n.v[2] = u[3] * inv_rho;
#pragma unroll
        for (int d = 0; d < 3; ++d) n.B[d] = u[5 + d];
        n.psi = u[8];
        n.p = P.gm1 * (u[4] - R(0.5) * (u[1] * n.v[0] + u[2] * n.v[1] + u[3] * n.v[2]) -
                       R(0.5) * (u[5] * u[5] + u[6] * u[6] + u[7] * u[7]) - R(0.5) * u[8] * u[8]);
        n.inv_gm1 = P.inv_gm1;
        if (LOGS) {
            n.lrho = node_log((L)n.rho);
            n.lp = node_log((L)n.p);
        } else {
            n.lrho = n.lp = 0.0;
        }
        return n;
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        f[0] = n.rho;
#pragma unroll
        for (int d = 0; d < 3; ++d) f[1 + d] = n.v[d];
        f[4] = n.p;
#pragma unroll
        for (int d = 0; d < 3; ++d) f[5 + d] = n.B[d];
        f[8] = n.psi;
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L lrho, L lp, const PhysR<R>& P) {
        Node<R, L> n;
        n.rho = f[0];
#pragma unroll
        for (int d = 0; d < 3; ++d) n.v[d] = f[1 + d];
        n.p = f[4];
#pragma unroll
        for (int d = 0; d < 3; ++d) n.B[d] = f[5 + d];
        n.psi = f[8];
        n.lrho = lrho;
        n.lp = lp;
        n.inv_gm1 = P.inv_gm1;
        return n;
    }

    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
        const R rho = n.rho;
        const R* v = n.v;
        const R* B = n.B;
        const R psi = n.psi;
        const R kin_en = R(0.5) * rho * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        const R mag_en = R(0.5) * (B[0] * B[0] + B[1] * B[1] + B[2] * B[2]);
        const R p_over_gm1 = n.p * P.inv_gm1;
        const R p = n.p;
        const R vB = v[0] * B[0] + v[1] * B[1] + v[2] * B[2];
        const R rho_vo = rho * v[o];
        f[0] = rho_vo;
#pragma unroll
        for (int d = 0; d < 3; ++d)
            f[1 + d] = (d == o) ? rho_vo * v[d] + p + mag_en - B[o] * B[o] : rho_vo * v[d] - B[o] * B[d];
        f[4] = (kin_en + P.gamma * p_over_gm1 + R(2) * mag_en) * v[o] - B[o] * vB + P.c_h * psi * B[o];
#pragma unroll
        for (int d = 0; d < 3; ++d) f[5 + d] = (d == o) ? P.c_h * psi : v[o] * B[d] - v[d] * B[o];
        f[8] = P.c_h * B[o];
    }

    // The argument of the fast speed's inner root, (a2 + b2)^2 - 4 a2 bo2 with
    // b2 = bo2 + bt2 (the field along and across the direction).  It is zero where
    // the field lies along the direction and a2 = b2, and the difference then rounds
    // below zero (in half of such states with a fused multiply-add), whose root is
    // NaN.  FP64: as a sum of squares.  FP32 arithmetic: the difference, kept from
    // falling below zero (the sum takes more registers than the spilling kernels on
    // refined meshes have: 3D RK stage at 4544 elements 106.5 -> 112 us).
    template <typename R>
    __device__ static R fast_root2(R a2, R b2, R bo2, R bt2) {
        if constexpr (std::is_same<R, double>::value) {
            const R d = a2 - b2;
            return d * d + R(4) * a2 * bt2;
        } else {
            const R s = a2 + b2;
            return dmax(s * s - R(4) * a2 * bo2, R(0));  // (a NaN stays)
        }
    }
    // |B|^2 across direction o
    template <typename R>
    __device__ static R transverse2(const R* B, int o) {
        R t = R(0);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            if (d != o) t += B[d] * B[d];
        return t;
    }
    template <typename R, typename L>
    __device__ static R fast_speed(const Node<R, L>& n, int o, const PhysR<R>& P) {
        const R inv_rho = rdiv(R(1), n.rho);
        const R a_square = P.gamma * n.p * inv_rho;
        const R t = transverse2(n.B, o);
        const R b_square = (std::is_same<R, double>::value
                                ? n.B[o] * n.B[o] + t
                                : n.B[0] * n.B[0] + n.B[1] * n.B[1] + n.B[2] * n.B[2]) * inv_rho;
        const R D = fast_root2(a_square, b_square, n.B[o] * n.B[o] * inv_rho, t * inv_rho);
        return rsqrt_(R(0.5) * (a_square + b_square) + R(0.5) * rsqrt_(D));
    }

    // Roe-averaged normal velocity and fast magnetoacoustic speed (Cargo &
    // Gallice 1997): weights sqrt(rho) / (sqrt(rho_l) + sqrt(rho_r)) for v, B
    // and the total enthalpy H = (rho e + p + |B|^2/2) / rho, the jump term
    // X = |[[B]]|^2 / (2 (sqrt(rho_l) + sqrt(rho_r))^2), b^2 = |B|^2 / sqrt(rho_l rho_r),
    // a^2 = (2 - gamma) X + (gamma - 1)(H - |v|^2/2 - b^2)
    template <typename R, typename L>
    __device__ static void roe_fast_speed(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R& vel,
                                          R& cf) {
        const R sl = rsqrt_(l.rho), sr = rsqrt_(r.rho);
        const R inv_add = rdiv(R(1), sl + sr), inv_prod = rdiv(R(1), sl * sr);
        const R wl = sl * inv_add, wr = sr * inv_add;
        R v2 = R(0), B2 = R(0), Bt2 = R(0), dB2 = R(0), Bo = R(0);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const R vd = l.v[d] * wl + r.v[d] * wr;
            const R Bd = l.B[d] * wl + r.B[d] * wr;
            const R db = l.B[d] - r.B[d];
            v2 += vd * vd;
            B2 += Bd * Bd;
            dB2 += db * db;
            if (d == o) {
                vel = vd;
                Bo = Bd;
            } else {
                Bt2 += Bd * Bd;
            }
        }
        const R mbl = l.B[0] * l.B[0] + l.B[1] * l.B[1] + l.B[2] * l.B[2];
        const R mbr = r.B[0] * r.B[0] + r.B[1] * r.B[1] + r.B[2] * r.B[2];
        const R Hl = rdiv(l.cons(4) + l.p + R(0.5) * mbl, l.rho), Hr = rdiv(r.cons(4) + r.p + R(0.5) * mbr, r.rho);
        const R H = Hl * wl + Hr * wr;
        const R X = R(0.5) * dB2 * inv_add * inv_add;
        const R b2 = (std::is_same<R, double>::value ? Bo * Bo + Bt2 : B2) * inv_prod;
        const R a2 = (R(2) - P.gamma) * X + P.gm1 * (H - R(0.5) * v2 - b2);
        const R astar = rsqrt_(fast_root2(a2, b2, Bo * Bo * inv_prod, Bt2 * inv_prod));
        cf = rsqrt_(R(0.5) * (a2 + b2 + astar));
    }

    // flux_hindenlang_gassner from its logarithmic means
    template <typename R, typename L>
    __device__ static void hindenlang_gassner(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P,
                                              R rho_mean, R inv_rho_p_mean, R* f) {
        const R* Bl = l.B;
        const R* Br = r.B;
        const R psil = l.psi, psir = r.psi;
        R vavg[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) vavg[d] = R(0.5) * (l.v[d] + r.v[d]);
        const R p_avg = R(0.5) * (l.p + r.p);
        const R psi_avg = R(0.5) * (psil + psir);
        const R velocity_square_avg = R(0.5) * (l.v[0] * r.v[0] + l.v[1] * r.v[1] + l.v[2] * r.v[2]);
        const R magnetic_square_avg = R(0.5) * (Bl[0] * Br[0] + Bl[1] * Br[1] + Bl[2] * Br[2]);
        const R f1 = rho_mean * vavg[o];
        f[0] = f1;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            R t = f1 * vavg[d];
            if (d == o) t = t + p_avg + magnetic_square_avg;
            f[1 + d] = t - R(0.5) * (Bl[o] * Br[d] + Br[o] * Bl[d]);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d)
            f[5 + d] = (d == o) ? P.c_h * psi_avg
                                : R(0.5) * (l.v[o] * Bl[d] - l.v[d] * Bl[o] + r.v[o] * Br[d] - r.v[d] * Br[o]);
        f[8] = P.c_h * R(0.5) * (Bl[o] + Br[o]);
        R s = l.p * r.v[o] + r.p * l.v[o];
#pragma unroll
        for (int d = 0; d < 3; ++d)
            if (d != o) s = s + (l.v[o] * Bl[d] * Br[d] + r.v[o] * Br[d] * Bl[d]);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            if (d != o) s = s - (l.v[d] * Bl[o] * Br[d] + r.v[d] * Br[o] * Bl[d]);
        s = s + P.c_h * (Bl[o] * psir + Br[o] * psil);
        f[4] = f1 * (velocity_square_avg + inv_rho_p_mean * P.inv_gm1) + R(0.5) * s;
    }

    // flux_hindenlang_gassner without node logarithms (FP64)
    template <int KIND, int MEANS, typename L>
    __device__ static void two_point_log_free(const Node<double, L>& l, const Node<double, L>& r, int o,
                                              const PhysR<double>& P, double* f) {
        static_assert(KIND == FLUX_HINDENLANG_GASSNER, "the flux with logarithmic means");
        double rho_mean, inv_mean;
        log_free_means<MEANS>(l.rho, r.rho, l.rho * r.p, r.rho * l.p, rho_mean, inv_mean);
        hindenlang_gassner(l, r, o, P, rho_mean, l.p * r.p * inv_mean, f);
    }
    // Local Lax-Friedrichs in FP64.  The physical flux is v_o u plus pressure
    // and magnetic terms (B_o and psi: c_h psi and c_h B_o alone), so that
    //   2 f = v_l,o u_l + v_r,o u_r + lambda (u_l - u_r) + those terms,
    // with |B|^2 shared by the fluxes, the states and the fast speeds.
    // (The interfaces are the heaviest part of the MHD kernel: 3D rhs! at 4096
    // elements 23.8 -> 23.3 us against two fluxes and two states.  1 / rho without
    // the quotient's residual step, which rounds nothing differently here: 23.5.)
    template <int KIND, typename L>
    __device__ static void lax_friedrichs(const Node<double, L>& l, const Node<double, L>& r, int o,
                                          const PhysR<double>& P, double* f) {
        const Node<double, L>* n[2] = {&l, &r};
        double u[2][9], c[2], en[2], pt[2], cB[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const double* v = n[k]->v;
            const double* B = n[k]->B;
            const double psi = n[k]->psi, p = n[k]->p;
            const double bt2 = transverse2(B, o), b2 = fma(B[o], B[o], bt2);
            u[k][0] = n[k]->rho;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                u[k][1 + d] = n[k]->rho * v[d];
                u[k][5 + d] = B[d];
            }
            u[k][8] = psi;
            const double mv = fma(u[k][3], v[2], fma(u[k][2], v[1], u[k][1] * v[0]));
            const double e = fma(p, P.inv_gm1, 0.5 * (mv + b2));  // without psi^2 / 2
            u[k][4] = fma(0.5 * psi, psi, e);
            pt[k] = fma(0.5, b2, p);
            cB[k] = P.c_h * B[o];
            const double vB = fma(v[2], B[2], fma(v[1], B[1], v[0] * B[0]));
            en[k] = fma(v[o], e + pt[k], fma(psi, cB[k], -(B[o] * vB)));
            const double ir = rrcp(n[k]->rho), as = P.gamma * p * ir, bs = b2 * ir;
            c[k] = rsqrt_(0.5 * (as + bs + rsqrt_(fast_root2(as, bs, 0.0, bt2 * ir))));
        }
        double lam;
        if (KIND == FLUX_LLF_NAIVE)
            lam = dmax(dabs(l.v[o]), dabs(r.v[o])) + dmax(c[0], c[1]);
        else
            lam = dmax(dabs(l.v[o]) + c[0], dabs(r.v[o]) + c[1]);
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            double t;
            if (q == 4) {
                t = en[0] + en[1];
            } else if (q == 5 + o) {
                t = P.c_h * (l.psi + r.psi);
            } else if (q == 8) {
                t = cB[0] + cB[1];
            } else if (q == 0) {
                t = u[0][1 + o] + u[1][1 + o];
            } else if (q <= 3) {
                t = fma(l.v[o], u[0][q], r.v[o] * u[1][q]);
                t = fma(-l.B[o], l.B[q - 1], fma(-r.B[o], r.B[q - 1], t));
                if (q == 1 + o) t += pt[0] + pt[1];
            } else {
                t = fma(l.v[o], u[0][q], r.v[o] * u[1][q]);
                t = fma(-l.v[q - 5], l.B[o], fma(-r.v[q - 5], r.B[o], t));
            }
            f[q] = 0.5 * fma(lam, u[0][q] - u[1][q], t);
        }
    }
    // whether every pair of these nodes satisfies MEANS_NEAR: rho, and rho / p
    // (v_rcp_f64 as it is: within 2^-24, far inside the polynomials' margin); false
    // for a node that is not a number
    template <int N, typename L>
    __device__ static bool near_line(const Node<double, L>* n) {
        double r0 = n[0].rho, r1 = r0, b0 = r0 * __builtin_amdgcn_rcp(n[0].p), b1 = b0, sum = n[0].p;
#pragma unroll
        for (int i = 1; i < N; ++i) {
            const double b = n[i].rho * __builtin_amdgcn_rcp(n[i].p);
            r0 = raw_min(r0, n[i].rho);
            r1 = raw_max(r1, n[i].rho);
            b0 = raw_min(b0, b);
            b1 = raw_max(b1, b);
            sum += n[i].p;
        }
        const bool a = near_ratio(r0, r1), b = near_ratio(b0, b1) && sum < 0x1p1000;
        return a && b && near_range(n[0].rho, n[0].p);
    }

    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        if constexpr (KIND == FLUX_HINDENLANG_GASSNER) {
            const R rho_mean = ln_mean_logs<R>(l.rho, r.rho, l.lrho, r.lrho);
            const R inv_rho_p_mean =
                l.p * r.p * inv_ln_mean_logs<R>(l.rho * r.p, r.rho * l.p, l.lrho + r.lp, r.lrho + l.lp);
            hindenlang_gassner(l, r, o, P, rho_mean, inv_rho_p_mean, f);
        } else if constexpr (std::is_same<R, double>::value && (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE)) {
            lax_friedrichs<KIND>(l, r, o, P, f);
        } else {
            R fl[9], fr[9];
            flux(l, o, P, fl);
            flux(r, o, P, fr);
            if (KIND == FLUX_LLF || KIND == FLUX_LLF_NAIVE) {
                const R cl = fast_speed(l, o, P), cr = fast_speed(r, o, P);
                R lam;
                if (KIND == FLUX_LLF_NAIVE)
                    lam = dmax(dabs(l.v[o]), dabs(r.v[o])) + dmax(cl, cr);
                else
                    lam = dmax(dabs(l.v[o]) + cl, dabs(r.v[o]) + cr);
                const R hl = R(-0.5) * lam;
#pragma unroll
                for (int q = 0; q < 9; ++q) f[q] = R(0.5) * (fl[q] + fr[q]) + hl * (r.cons(q) - l.cons(q));
            } else if (KIND == FLUX_HLLE) {
                // HLL with Einfeldt's estimates: the states' fast speeds and the
                // Roe-averaged fast speed of Cargo & Gallice (1997)
                R vroe, croe;
                roe_fast_speed(l, r, o, P, vroe, croe);
                const R a = l.v[o] - fast_speed(l, o, P), b = vroe - croe;
                const R cc = r.v[o] + fast_speed(r, o, P), dd = vroe + croe;
                const R lmin = b < a ? b : a;
                const R lmax = dmax(cc, dd);
                if (lmin >= R(0) && lmax >= R(0)) {
#pragma unroll
                    for (int q = 0; q < 9; ++q) f[q] = fl[q];
                } else if (lmax <= R(0) && lmin <= R(0)) {
#pragma unroll
                    for (int q = 0; q < 9; ++q) f[q] = fr[q];
                } else {
                    const R inv = rdiv(R(1), lmax - lmin);
                    const R fll = lmax * inv, frr = lmin * inv, fdiss = lmin * lmax * inv;
#pragma unroll
                    for (int q = 0; q < 9; ++q) f[q] = fll * fl[q] - frr * fr[q] + fdiss * (r.cons(q) - l.cons(q));
                }
            } else {
#pragma unroll
                for (int q = 0; q < 9; ++q) f[q] = R(0.5) * (fl[q] + fr[q]);
            }
        }
    }

    // flux_nonconservative_powell(u_ll, u_rr, o): Powell (0, B, v.B, v, 0) and
    // Galilean GLM terms of the left state times the right state's B_o / psi.
    template <int POS, typename R, typename L>
    __device__ static void noncons(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>&, R* f) {
        const R v_dot_B_ll = l.v[0] * l.B[0] + l.v[1] * l.B[1] + l.v[2] * l.B[2];
        const R Bo_rr = r.B[o];
        const R psi_rr = r.psi;
        const R psi_vo_ll = l.psi * l.v[o];
        f[0] = R(0);
#pragma unroll
        for (int d = 0; d < 3; ++d) f[1 + d] = l.B[d] * Bo_rr;
        f[4] = v_dot_B_ll * Bo_rr + psi_vo_ll * psi_rr;
#pragma unroll
        for (int d = 0; d < 3; ++d) f[5 + d] = l.v[d] * Bo_rr;
        f[8] = l.v[o] * psi_rr;
    }

    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        const R rho = u[0];
        const R v1 = u[1] / rho, v2 = u[2] / rho, v3 = u[3] / rho;
        const R B1 = u[5], B2 = u[6], B3 = u[7], psi = u[8];
        const R kin_en = R(0.5) * rho * (v1 * v1 + v2 * v2 + v3 * v3);
        const R mag_en = R(0.5) * (B1 * B1 + B2 * B2 + B3 * B3);
        const R p = P.gm1 * (u[4] - kin_en - mag_en - R(0.5) * psi * psi);
        const R a_square = P.gamma * p / rho;
        const R sqrt_rho = sqrt(rho);
        const R b1 = B1 / sqrt_rho, b2 = B2 / sqrt_rho, b3 = B3 / sqrt_rho;
        const R b_square = b1 * b1 + b2 * b2 + b3 * b3;
        const R vv[3] = {v1, v2, v3}, bb[3] = {b1, b2, b3};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const R s = a_square + b_square;
            const R cf = sqrt(R(0.5) * s + R(0.5) * sqrt(fast_root2(a_square, b_square, R(0), transverse2(bb, d))));
            lam[d] = dabs(vv[d]) + cf;
        }
    }
};

// ===========================================================================
// Ideal MHD in 1D (Trixi IdealGlmMhdEquations1D): (rho, rho v1..3, rho e,
// B1..3), no cleaning field and no nonconservative terms (B1 is constant).
// The GLM-MHD fluxes with psi = 0 and c_h = 0 (the host sets c_h = 0 for 1D)
// are its fluxes, so this wraps them with the cleaning field held at zero.
// ===========================================================================
struct GlmMhd1D {
    static constexpr int NV = 8;
    static constexpr bool NONCONS = false;
    static constexpr int NRF = GlmMhd::NRF;
    template <typename R, typename L = R>
    using Node = GlmMhd::Node<R, L>;
    template <typename R, bool LOGS, typename L = R>
    __device__ static Node<R, L> node(const R* u, const PhysR<R>& P) {
        R u9[9];
#pragma unroll
        for (int q = 0; q < 8; ++q) u9[q] = u[q];
        u9[8] = R(0);
        return GlmMhd::template node<R, LOGS, L>(u9, P);
    }
    template <typename R, typename L>
    __device__ static void to_rec(const Node<R, L>& n, R* f) {
        GlmMhd::to_rec(n, f);
    }
    template <typename R, typename L>
    __device__ static Node<R, L> from_rec(const R* f, L lrho, L lp, const PhysR<R>& P) {
        return GlmMhd::from_rec(f, lrho, lp, P);
    }
    template <typename R, typename L>
    __device__ static void flux(const Node<R, L>& n, int o, const PhysR<R>& P, R* f) {
        R f9[9];
        GlmMhd::flux(n, o, P, f9);
#pragma unroll
        for (int q = 0; q < 8; ++q) f[q] = f9[q];
    }
    template <int KIND, typename R, typename L>
    __device__ static void two_point(const Node<R, L>& l, const Node<R, L>& r, int o, const PhysR<R>& P, R* f) {
        R f9[9];
        GlmMhd::template two_point<KIND>(l, r, o, P, f9);
#pragma unroll
        for (int q = 0; q < 8; ++q) f[q] = f9[q];
    }
    template <int POS, typename R, typename L>
    __device__ static void noncons(const Node<R, L>&, const Node<R, L>&, int, const PhysR<R>&, R* f) {
#pragma unroll
        for (int q = 0; q < 8; ++q) f[q] = R(0);
    }
    template <typename R>
    __device__ static void max_abs_speeds(const R* u, const PhysR<R>& P, R* lam) {
        R u9[9];
#pragma unroll
        for (int q = 0; q < 8; ++q) u9[q] = u[q];
        u9[8] = R(0);
        GlmMhd::max_abs_speeds(u9, P, lam);
    }
};

// FP64 kernels of compressible Euler whose fluxes all have a doubled form
// (twice_flux): they accumulate twice every term and halve once at the end.
template <class EQ>
struct IsEuler : std::false_type {};
template <int DIM>
struct IsEuler<Euler<DIM>> : std::true_type {};
constexpr bool twice_kind(int k) {
    return k == FLUX_RANOCHA || k == FLUX_SHIMA_ETAL || k == FLUX_LLF || k == FLUX_LLF_NAIVE;
}
template <class EQ, typename R, int VOL, int VF, int SF, int FVF>
constexpr bool twice_fluxes() {
    return IsEuler<EQ>::value && std::is_same<R, double>::value && VOL != VI_WEAK && twice_kind(VF) &&
           twice_kind(SF) && (VOL != VI_HG || twice_kind(FVF));
}
// FP64 kernels that take the logarithmic means without node logarithms
// (every Euler kernel with such a flux has the doubled form).
template <class EQ, typename R, bool TWICE>
constexpr bool log_free() {
    return TWICE || (std::is_same<EQ, GlmMhd>::value && std::is_same<R, double>::value);
}

// Two-point flux: twice the flux where TWICE (ul, ur: the conservative states
// of the nodes, read by the Lax-Friedrichs kinds only), otherwise from nodes
// that carry logarithms where their flux and arithmetic type need them.
template <class EQ, int KIND, bool TWICE, int MEANS, typename R, typename L>
__device__ __forceinline__ void node_flux(const typename EQ::template Node<R, L>& l, const R* ul,
                                          const typename EQ::template Node<R, L>& r, const R* ur, int o,
                                          const PhysR<R>& P, R* f) {
    if constexpr (TWICE)
        EQ::template twice_flux<KIND, MEANS>(l, ul, r, ur, o, P, f);
    else if constexpr (MEANS != MEANS_LOGS && log_free<EQ, R, TWICE>() && flux_needs_logs(KIND))
        EQ::template two_point_log_free<KIND, MEANS>(l, r, o, P, f);
    else
        EQ::template two_point<KIND>(l, r, o, P, f);
}
// whether a node_flux of this kind reads the conservative states
constexpr bool flux_reads_cons(bool twice, int k) { return twice && (k == FLUX_LLF || k == FLUX_LLF_NAIVE); }

}  // namespace trixi_hip
