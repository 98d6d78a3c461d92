// vjp_group_kernel.hpp -- the adjoint of rhs! (FP64 flux differencing in 2D and
// 3D) in the lane groups of rhs_group_kernel: group d < DIM takes the volume
// pairs of the lines in direction d, the last group the interfaces of every
// direction, and the final pass has one lane per node.
//
// What bounded the form with one lane per line: its nodes, logarithms and
// cotangents in registers left one wave per SIMD, which waited for half of its
// time.  Here a lane keeps only its sums and reads a pair's nodes and cotangents
// from LDS, so that four waves per SIMD fit (128 registers); node_place keeps
// those reads free of bank conflicts, log_free_mean_grads needs no logarithms,
// and the volume code has its direction as a constant, so that field offsets are
// part of the load instructions.  What is left is FP64 issue (34 million wave
// instructions at 32768 elements, half of the VALU's slots at 105 us on one pair of
// buffers) and the waits of a workgroup's first pass and barriers.
//
// 3D Euler at 32768 elements 168 -> 124 us (136 with the direction as data, 130
// before the fluxes' adjoints were shortened; tiles of 4 elements 143); 2D Euler
// at 65536 elements 60.4 -> 43; floor of its bytes 51 us in 3D.
#pragma once

#include "launch_rhs.hpp"
#include "vjp_kernel.hpp"

namespace trixi_hip {

template <class EQ>
struct VjpRotation;
template <int DIM>
struct VjpRotation<EulerVjp<DIM>> {
    // position of variable (or record field) k of a vector read from component o on
    __device__ static int variable(int k, int o) { return rotated(k, 1, DIM, o); }
};

// Place of a node in the LDS arrays (N = 4): its first index is exchanged with
// the others', so that the lines of every direction lie in different banks.
template <int N>
__device__ __forceinline__ int node_place(int n) {
    return N == 4 ? n ^ ((n >> 2) & 3) : n;
}

// WAVES: waves per SIMD the registers are allocated for
template <int DIM, int N, class EQ, int VF, int SF, int M, bool EXT, int WAVES>
__global__ void __launch_bounds__((group_threads<DIM, N, M>()), WAVES) vjp_group_kernel(const VjpArgs a) {
    constexpr int NL = cpow(N, DIM - 1);
    constexpr int NN = cpow(N, DIM);
    constexpr int GL = M * NL;  // lanes of a group
    constexpr int NT = GL * (DIM + 1);
    constexpr int NIT = (NN * M + NT - 1) / NT;  // nodes per lane of the node and final passes
    constexpr int NV = EQ::NV;
    constexpr int NRG = NV + 1;  // node record: rho, v, p, c
    static_assert(GL % 64 == 0 && NT % M == 0 && !EQ::NONCONS, "whole waves per group, conservative equations");
    using Node = typename EQ::template Node<double>;
    using Bar = typename EQ::template Bar<double>;
    using Rot = VjpRotation<EQ>;

    // node records (later the sums of direction 1), scaled cotangents (later
    // the sums of the other directions), face cotangents
    // [direction][side][line][variable]
    __shared__ double rec[NRG * NN * M];
    __shared__ double ws[NV * NN * M];
    __shared__ double fcs[DIM * 2 * NL * NV * M];

    const int tid = threadIdx.x;
    const int grp = __builtin_amdgcn_readfirstlane(tid / GL);
    const int el = tid % M;
    const int line = (tid / M) % NL;
    const int64_t E = a.E;
    const uint32_t E32 = (uint32_t)E;
    const int64_t slab = (int64_t)NN * E;
    const int64_t e0 = xcd_tile(a.nxcd) * M;
    if (e0 >= E) return;  // whole workgroup: padding tile of the XCD mapping
    const int64_t ec = e0 + el < E ? e0 + el : E - 1;
    const PhysR<double> P = PhysR<double>::from(a.phys);

    const bool faces = grp == DIM;
    // neighbours of direction 0, then of the direction after the current one
    int32_t nm = 0, np = 0;
    auto load_neighbours = [&](int o) {
        nm = a.nbr[(int64_t)(2 * o) * E + ec];
        np = a.nbr[(int64_t)(2 * o + 1) * E + ec];
    };
    if (faces) load_neighbours(0);

    // this lane's nodes of the node pass, requested before anything waits
    double un[NIT][NV], vn[NIT][NV];
    const double invj = a.invJ[ec];  // (a lane's nodes are of its own element)
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        int q = tid + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) q = NN * M - 1;
        const int64_t ee = e0 + q % M < E ? e0 + q % M : E - 1;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t g = soa(v, q / M, ee, slab, E32);
            un[it][v] = a.u[g];
            vn[it][v] = a.vbar[g];
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    auto first_node = [&](int o) {
        return o == 0 ? line_base<DIM, N>(line, 0) : (o == 1 ? line_base<DIM, N>(line, 1) : line_base<DIM, N>(line, 2));
    };
    // state and cotangent of a neighbour's face node, rotated
    struct Side {
        double u[NV], vb[NV], invj;
        bool boundary;
    };
    auto load_side = [&](int o, bool plus, int32_t n, Side& x) {
        const int s = o == 0 ? 1 : (o == 1 ? N : N * N);
        x.boundary = EXT && n < 0;  // its loads read this element
        if (x.boundary) n = (int32_t)ec;
        const int node = first_node(o) + (plus ? 0 : (N - 1) * s);
        x.invj = a.invJ[n];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t g = soa(Rot::variable(v, o), node, n, slab, E32);
            x.u[v] = a.u[g];
            x.vb[v] = a.vbar[g];
        }
    };

    // ---- node pass ---------------------------------------------------------
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        int q = tid + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) continue;
        q = node_place<N>(q / M) * M + q % M;
        const Node n = EQ::template node<double, false>(un[it], P);
        rec[q] = n.rho;
#pragma unroll
        for (int d = 0; d < DIM; ++d) rec[(1 + d) * NN * M + q] = n.v[d];
        rec[(DIM + 1) * NN * M + q] = n.p;
        rec[(DIM + 2) * NN * M + q] = n.c;
        const double wsc = -invj * a.alpha;
#pragma unroll
        for (int v = 0; v < NV; ++v) ws[v * NN * M + q] = wsc * vn[it][v];
    }
    __syncthreads();

    auto slot = [&](int node) { return node_place<N>(node) * M + el; };
    auto staged = [&](int q, int o) {
        double f[NRG];
#pragma unroll
        for (int k = 0; k < NRG; ++k) f[k] = rec[Rot::variable(k, o) * NN * M + q];
        return EQ::from_short_rec(f);
    };
    auto cotangent = [&](int q, int o, double* w) {
#pragma unroll
        for (int v = 0; v < NV; ++v) w[v] = ws[Rot::variable(v, o) * NN * M + q];
    };

    Bar bb[N];
    int sl[N];  // the line's nodes
    // ---- volume terms of one direction (a constant: the fields' offsets are
    // then part of the load instructions) ------------------------------------
    auto volume = [&](auto dc) {
        constexpr int o = decltype(dc)::value;
#pragma unroll
        for (int p = 0; p < N; ++p) sl[p] = slot(line_base<DIM, N>(line, o) + p * cpow(N, o));
#pragma unroll
        for (int p = 0; p < N; ++p) EQ::zero(bb[p]);
        // the series means of every pair; a wave in which some line has a jump
        // of more than a third takes one pair per turn with its checks
        bool near = true;
        if constexpr (flux_needs_logs(VF)) {
            Node nd[N];
#pragma unroll
            for (int p = 0; p < N; ++p) nd[p] = staged(sl[p], o);
            near = __builtin_amdgcn_ballot_w64(!Euler<DIM>::template near_line<N>(nd)) == 0;
        }
        auto pair = [&](int i, int j, auto means, Bar& bi, Bar& bj) {
            // the means from densities and pressures first, the rest read after
            // them, and read again for each pair (registers)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            int ni = sl[0], nj = sl[0];
#pragma unroll
            for (int p = 1; p < N; ++p) {
                ni = i == p ? sl[p] : ni;
                nj = j == p ? sl[p] : nj;
            }
            double rl = 0.0, dLx = 0.0, dLy = 0.0, I = 0.0, dIx = 0.0, dIy = 0.0;
            if constexpr (VF == FLUX_RANOCHA) {
                const double ri = rec[ni], rj = rec[nj];
                const double pi = rec[(DIM + 1) * NN * M + ni], pj = rec[(DIM + 1) * NN * M + nj];
                log_free_mean_grads<decltype(means)::value>(ri, rj, ri * pj, rj * pi, rl, dLx, dLy, I, dIx, dIy);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            constexpr double half = VF == FLUX_RANOCHA ? 0.5 : 1.0;
            const double fa = half * a.Ds[i * N + j], fb = half * a.Ds[j * N + i];
            double g[NV], w[NV];
            cotangent(ni, o, g);
            cotangent(nj, o, w);
#pragma unroll
            for (int v = 0; v < NV; ++v) g[v] = fa * g[v] + fb * w[v];
            const Node l = staged(ni, o), r = staged(nj, o);
            if constexpr (VF == FLUX_RANOCHA)
                EQ::ranocha_vjp(l, r, 0, g, bi, bj, P, rl, dLx, dLy, I, dIx, dIy);
            else
                EQ::template two_point_vjp<VF>(l, r, 0, g, bi, bj, P);
        };
        if (near) {
#pragma unroll
            for (int i = 0; i < N; ++i)
#pragma unroll
                for (int j = i + 1; j < N; ++j) pair(i, j, std::integral_constant<int, MEANS_NEAR>{}, bb[i], bb[j]);
        } else {
#pragma unroll 1
            for (int i = 0; i + 1 < N; ++i)
#pragma unroll 1
                for (int j = i + 1; j < N; ++j) {
                    Bar bi, bj;
                    EQ::zero(bi);
                    EQ::zero(bj);
                    pair(i, j, std::integral_constant<int, MEANS_ANY>{}, bi, bj);
                    double ti[NV], tj[NV];
                    EQ::bar_to_array(bi, ti);
                    EQ::bar_to_array(bj, tj);
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        double t[NV];
                        EQ::bar_to_array(bb[p], t);
#pragma unroll
                        for (int v = 0; v < NV; ++v) t[v] += p == i ? ti[v] : (p == j ? tj[v] : 0.0);
                        EQ::array_to_bar(t, bb[p]);
                    }
                }
        }
    };
    if (grp == 0) volume(std::integral_constant<int, 0>{});
    if (grp == 1) volume(std::integral_constant<int, 1>{});
    if constexpr (DIM > 2) {
        if (grp == 2) volume(std::integral_constant<int, 2>{});
    }
    if (faces) {
        // ---- interfaces of every direction, one after the other ----------------
        auto face = [&](int o, bool plus, Side& x) {
            const int so = o == 0 ? 1 : (o == 1 ? N : N * N);
            const int node = first_node(o) + (plus ? (N - 1) * so : 0);
            double g[NV];
            cotangent(slot(node), o, g);
            const double lo = plus ? a.lhat_p : -a.lhat_m;
            double ln = (plus ? -a.lhat_m : a.lhat_p) * (-x.invj * a.alpha);
            if constexpr (EXT) {
                // a Dirichlet state does not depend on u and has no cotangent
                if (x.boundary) {
                    ln = 0.0;
                    double xx[3] = {0.0, 0.0, 0.0}, uu[5];
#pragma unroll
                    for (int dd = 0; dd < DIM; ++dd) xx[dd] = a.x[((int64_t)dd * NN + node) * E + ec];
                    boundary_value(a.bc_ic, xx, a.t, uu);
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const int w = Rot::variable(v, o);
#pragma unroll
                        for (int q = 0; q < NV; ++q)
                            if (q == w) x.u[v] = uu[q];
                        x.vb[v] = 0.0;
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) g[v] = lo * g[v] + ln * x.vb[v];
            const Node nbn = EQ::template node<double, false>(x.u, P);
            const Node own = staged(slot(node), o);
            Bar b;
            EQ::zero(b);
            if (plus)
                EQ::template own_side_vjp<SF, false>(own, nbn, x.u, 0, g, b, P);
            else
                EQ::template own_side_vjp<SF, true>(own, nbn, x.u, 0, g, b, P);
            double t[NV];
            EQ::bar_to_array(b, t);
#pragma unroll
            for (int v = 0; v < NV; ++v)
                fcs[(((2 * o + (plus ? 1 : 0)) * NL + line) * NV + Rot::variable(v, o)) * M + el] = t[v];
        };
#pragma unroll
        for (int o = 0; o < DIM; ++o) {
            Side sm, sp;
            load_side(o, false, nm, sm);
            load_side(o, true, np, sp);
            if (o + 1 < DIM) load_neighbours(o + 1);
            face(o, false, sm);
            __builtin_amdgcn_sched_barrier(0);
            face(o, true, sp);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // the lane index anew: its uses below would otherwise keep the node pass's
    // addresses in registers through the fluxes
    int tid2 = tid;
    asm volatile("" : "+v"(tid2));
    // the node's state and what the outputs need, requested before the sums meet
    double uu[NIT][NV], prev[NIT][NV], vb2[NIT][NV];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        int q = tid2 + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) q = NN * M - 1;
        const int64_t ee = e0 + q % M < E ? e0 + q % M : E - 1;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t g = soa(v, q / M, ee, slab, E32);
            uu[it][v] = a.u[g];
            prev[it][v] = a.beta != 0.0 ? a.beta * a.ubar[g] : 0.0;
            vb2[it][v] = a.kbar_out != nullptr ? a.vbar[g] : 0.0;
        }
    }
    __syncthreads();
    // direction 0 into the cotangents' place, direction 1 into the records',
    // direction 2 added to direction 0
    auto put = [&](double* dst, bool add) {
#pragma unroll
        for (int p = 0; p < N; ++p) {
            double t[NV];
            EQ::bar_to_array(bb[p], t);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                double& x = dst[Rot::variable(v, grp) * NN * M + sl[p]];
                x = add ? x + t[v] : t[v];
            }
        }
    };
    if (grp == 0) put(ws, false);
    if (grp == 1) put(rec, false);
    __syncthreads();
    if constexpr (DIM > 2) {
        if (grp == 2) put(ws, true);
        __syncthreads();
    }

    // ---- final pass: the node's sum into conservative space, the outputs -----
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const int q = tid2 + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) continue;
        const int c = q % M, n = q / M;
        const int64_t e = e0 + c;
        if (e >= E) continue;
        const int ql = node_place<N>(n) * M + c;
        double t[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) t[v] = ws[v * NN * M + ql] + rec[v * NN * M + ql];
        int rest = n, idx[3] = {0, 0, 0};
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            idx[d] = rest % N;
            rest /= N;
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            // the node's line in direction d: its other indices, first fastest
            int ln = 0, w = 1;
#pragma unroll
            for (int dd = 0; dd < DIM; ++dd) {
                if (dd == d) continue;
                ln += idx[dd] * w;
                w *= N;
            }
            if (idx[d] == 0 || idx[d] == N - 1) {
                const int side = idx[d] == 0 ? 0 : 1;
#pragma unroll
                for (int v = 0; v < NV; ++v) t[v] += fcs[(((2 * d + side) * NL + ln) * NV + v) * M + c];
            }
        }
        Bar tot;
        EQ::array_to_bar(t, tot);
        double ub[NV];
        EQ::to_cons_bar(EQ::template node<double, false>(uu[it], P), tot, ub, P);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t g = soa(v, n, e, slab, E32);
            const double ubn = prev[it][v] + ub[v];
            a.ubar[g] = ubn;
            // (vbar is not written by this kernel: the neighbours' reads of
            // it stay valid, kbar_out being another buffer)
            if (a.kbar_out != nullptr) a.kbar_out[g] = a.kbar_a * vb2[it][v] + a.kbar_b * ubn;
        }
    }
}

// Equations with a lane-group form of the adjoint.
template <class EQ>
struct HasVjpRotation : std::false_type {};
template <int DIM>
struct HasVjpRotation<EulerVjp<DIM>> : std::true_type {};
template <int DIM, int N, class EQ, int VOL>
constexpr bool vjp_group_eligible() {
    return DIM > 1 && VOL == VI_FD && HasVjpRotation<EQ>::value &&
           (group_elems<DIM, N, EQ::NV, EQ::NV + 1>() * cpow(N, DIM - 1)) % 64 == 0 &&
           group_threads<DIM, N, group_elems<DIM, N, EQ::NV, EQ::NV + 1>()>() <= 1024;
}

// M: elements per workgroup of the one-group form; MG: of the
// direction-group form, used for meshes whose one-group form would launch
// fewer lanes than a.pd_lanes (on 2D and 3D meshes).  The lane-group form takes
// the place of the one-group form where it is built, and from a quarter of the
// lanes on that of the direction-group form: kernel times in 3D 9.3 (direction
// groups) and 9.6 us at 512 elements, 23.5 and 17.8 at 4096; in 2D 7.3 and 7.6
// at 4096, 18.0 and 13.1 at 16384.
template <int DIM, int N, class EQ, int VOL, int VF, int SF, int FVF, typename R, int M, bool EXT = false,
          int MG = M>
hipError_t launch_vjp(const VjpArgs& a, hipStream_t stream) {
    constexpr int NL = cpow(N, DIM - 1);
    auto grid = [&](int m) {
        int64_t blocks = (a.E + m - 1) / m;
        if (a.nxcd > 1) blocks = (blocks + a.nxcd - 1) / a.nxcd * a.nxcd;
        return dim3((unsigned)blocks);
    };
    if constexpr (DIM > 1) {
        if (a.E * NL < (vjp_group_eligible<DIM, N, EQ, VOL>() ? a.pd_lanes / 4 : a.pd_lanes)) {
            hipLaunchKernelGGL((vjp_kernel<DIM, N, EQ, VOL, VF, SF, FVF, R, MG, EXT, DIM>), grid(MG),
                               dim3(MG * NL * vjp_groups<DIM, N, VOL, EQ::NV, EQ::NRF, DIM>()), 0, stream, a);
            return hipGetLastError();
        }
    }
    if constexpr (vjp_group_eligible<DIM, N, EQ, VOL>()) {
        constexpr int ME = group_elems<DIM, N, EQ::NV, EQ::NV + 1>();
        // half the elements and two waves per SIMD where four spill: boundary
        // faces, and logarithmic means at the interfaces (3D Euler at 32768
        // elements with flux_ranocha there 221 -> 142 us)
        constexpr bool HALF = EXT || flux_needs_logs(SF);
        constexpr int MV = HALF && (ME / 2 * NL) % 64 == 0 ? ME / 2 : ME;
        constexpr int W = HALF ? 2 : (DIM == 3 ? 4 : TRIXI_HIP_GROUP_WAVES2D);
        hipLaunchKernelGGL((vjp_group_kernel<DIM, N, EQ, VF, SF, MV, EXT, W>), grid(MV),
                           dim3(group_threads<DIM, N, MV>()), 0, stream, a);
    } else {
        hipLaunchKernelGGL((vjp_kernel<DIM, N, EQ, VOL, VF, SF, FVF, R, M, EXT, 1>), grid(M), dim3(M * NL), 0, stream,
                           a);
    }
    return hipGetLastError();
}

}  // namespace trixi_hip
