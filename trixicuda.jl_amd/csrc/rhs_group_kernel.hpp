// rhs_group_kernel.hpp -- the FP64 rhs! (and fused Runge-Kutta stage) of flux
// differencing and shock capturing in 2D and 3D: lane groups by kind of work.
//
// A workgroup owns M elements and has DIM + 1 lane groups of M * N^(DIM-1)
// lanes (whole waves).  Group d < DIM evaluates the volume terms of the lines
// in direction d, lane (el, line) one line; the last group evaluates the
// interface fluxes of every direction, lane (el, line) both ends of its line,
// direction after direction.  For N = 4 in 3D the two kinds of group do the
// same work (six two-point fluxes; six interface fluxes), and there is one
// lane per node, so that the node pass and the final pass take one node per
// lane.
//
// Why this split: what bounds the kernel on meshes larger than the caches is
// the width of its rows in memory (M elements of one variable and node are
// contiguous).  A copy of the state of 32768 elements (two 84 MB arrays, three
// pairs in turn) takes 68 us in rows of 4, 50 in rows of 8 and 42 in rows of
// 16 elements, whatever is computed; with one lane group per direction that
// also evaluates its own faces, 4 elements were the most that kept several
// workgroups per compute unit.  Taking the faces (and their neighbour states)
// out of the volume lanes leaves room for four waves per SIMD at M = 8.
//
// Measured against one lane group per direction (M = 4): three CFL steps of 3D
// Euler at 32768 elements 1985 -> 1720 us, five steps on a refined mesh of 960
// elements 807 -> 647 us, rhs! alone at 32768 elements 83.7 -> 81.0 us (with
// the device time loop, the constants behind a pointer and the loads ahead of
// the fluxes now 1530, 561 and 78.9 us).  An XOR exchange of the node places
// against the bank conflicts of x-lines (node_place in vjp_group_kernel.hpp)
// gained 1 % for MHD and cost 1 % here and 3 % in 2D.  A
// register spilled in this kernel costs more than everything else (each lane's
// scratch goes to memory: 44 bytes per lane, 82 -> 118 us), hence the shape of
// the code below: one face after the other, the lane index hidden from the
// compiler before the final pass, no node kept across the rare pair loop.
//
// The direction is data, not code: fields of a vector are read in rotated
// order (component o first), so every group runs the same instructions with
// o = 0, and sums are stored back through the same rotation.
#pragma once

#include "rhs_kernel.hpp"

namespace trixi_hip {

// Position of field k of a rotated node record (or of variable k of a rotated
// state) in the stored one: the components of a vector starting at `first`
// are read from component o on.
__device__ __forceinline__ int rotated(int k, int first, int len, int o) {
    if (k < first || k >= first + len) return k;
    const int c = k - first + o;
    return first + (c >= len ? c - len : c);
}
template <class EQ>
struct Rotation;
template <int DIM>
struct Rotation<Euler<DIM>> {
    __device__ static int field(int k, int o) { return rotated(k, 1, DIM, o); }
    __device__ static int variable(int k, int o) { return rotated(k, 1, DIM, o); }
};
template <>
struct Rotation<GlmMhd> {
    __device__ static int field(int k, int o) { return rotated(rotated(k, 1, 3, o), 5, 3, o); }
    __device__ static int variable(int k, int o) { return field(k, o); }
};

// The nonconservative volume terms of a line, sum_j D_split[i,j] nc(u_i, u_j):
// the Powell and GLM terms are products of the left node's fields with the
// right node's B_o and psi, so the sums over j are taken once per node.
template <int N>
__device__ __forceinline__ void line_noncons(const GlmMhd::Node<double, double> (&nd)[N], const double* Ds,
                                             double scale, double (&al)[N][GlmMhd::NV]) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        double sB = 0.0, sP = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            sB = fma(Ds[i * N + j], nd[j].B[0], sB);
            sP = fma(Ds[i * N + j], nd[j].psi, sP);
        }
        sB *= scale;
        sP *= scale;
        const double* v = nd[i].v;
        const double* B = nd[i].B;
        const double vB = fma(v[2], B[2], fma(v[1], B[1], v[0] * B[0]));
        const double w = v[0] * sP;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            al[i][1 + d] = fma(B[d], sB, al[i][1 + d]);
            al[i][5 + d] = fma(v[d], sB, al[i][5 + d]);
        }
        al[i][4] = fma(vB, sB, fma(nd[i].psi, w, al[i][4]));
        al[i][8] += w;
    }
}

template <int DIM, int N, int M>
__host__ __device__ constexpr int group_threads() {
    return M * cpow(N, DIM - 1) * (DIM + 1);
}

// WAVES: waves per SIMD the registers are allocated for
template <int DIM, int N, class EQ, int VOL, int VF, int SF, int FVF, int M, bool RK, bool EXT, int WAVES>
__global__ void __launch_bounds__((group_threads<DIM, N, M>()), WAVES) rhs_group_kernel(const RhsArgs a, const RhsConst* __restrict__ consts) {
    const RhsConst& kc = *consts;
    constexpr int NL = cpow(N, DIM - 1);
    constexpr int NN = cpow(N, DIM);
    constexpr int GL = M * NL;                   // lanes of a group
    constexpr int NT = GL * (DIM + 1);
    constexpr int NIT = (NN * M + NT - 1) / NT;  // nodes per lane of the node and final passes
    constexpr int NV = EQ::NV;
    constexpr int NRF = EQ::NRF;
    constexpr bool TW = twice_fluxes<EQ, double, VOL, VF, SF, FVF>();
    constexpr bool LF = log_free<EQ, double, TW>();
    constexpr bool VF_LOGS = flux_needs_logs(VF);
    static_assert(LF || !(VF_LOGS || flux_needs_logs(SF) || flux_needs_logs(FVF)), "no node logarithms here");
    static_assert(VOL != VI_WEAK && GL % 64 == 0 && NV <= NRF, "whole waves per group");
    using Node = typename EQ::template Node<double, double>;
    using Rot = Rotation<EQ>;
    const double* __restrict__ U = static_cast<const double*>(a.u);

    // node records (later the sums of direction 1), sums of directions 0 and 2,
    // weighted interface fluxes [direction][side][line][variable]
    __shared__ double rec[NRF * NN * M];
    __shared__ double acc[NV * NN * M];
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
    const PhysR<double> P = PhysR<double>::from(kc.phys);
    double tnow = 0.0;
    if constexpr (EXT) tnow = RK ? a.time[0] : a.t_host;

    // neighbours of the lane's element: read by the face group, and by every
    // group for the smoothing of the blending factor
    const bool faces = grp == DIM;
    int32_t nb[2 * DIM];
    if (VOL == VI_HG || faces) {
#pragma unroll
        for (int f = 0; f < 2 * DIM; ++f) nb[f] = a.nbr[(int64_t)f * E + ec];
    }

    // this lane's nodes of the node pass, requested before anything waits
    double un[NIT][NV];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        int q = tid + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) q = NN * M - 1;
        const int64_t ee = e0 + q % M < E ? e0 + q % M : E - 1;
#pragma unroll
        for (int v = 0; v < NV; ++v) un[it][v] = U[soa(v, q / M, ee, slab, E32)];
    }
    __builtin_amdgcn_sched_barrier(0);

    // neighbour face states of direction o (rotated), for the face group
    double um[NV], up[NV];
    auto load_faces = [&](int o, double* m, double* p) {
        const int s = o == 0 ? 1 : (o == 1 ? N : N * N);
        const int base = o == 0 ? line_base<DIM, N>(line, 0) : (o == 1 ? line_base<DIM, N>(line, 1) : line_base<DIM, N>(line, 2));
        int32_t nm = nb[0], np = nb[1];
#pragma unroll
        for (int f = 1; f < DIM; ++f) {
            nm = o == f ? nb[2 * f] : nm;
            np = o == f ? nb[2 * f + 1] : np;
        }
        if constexpr (EXT) {  // boundary and mortar faces read this element instead
            nm = nm < 0 ? (int32_t)ec : nm;
            np = np < 0 ? (int32_t)ec : np;
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int w = Rot::variable(v, o);
            m[v] = U[soa(w, base + (N - 1) * s, nm, slab, E32)];
            p[v] = U[soa(w, base, np, slab, E32)];
        }
    };
    if (faces) load_faces(0, um, up);

    if (RK && a.done != nullptr && *a.done != 0.0) return;  // uniform

    // ---- node pass ---------------------------------------------------------
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const int q = tid + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) continue;
        const Node n = EQ::template node<double, false, double>(un[it], P);
        double f[NRF];
        EQ::to_rec(n, f);
#pragma unroll
        for (int k = 0; k < NRF; ++k) rec[k * NN * M + q] = f[k];
    }
    __syncthreads();

    auto staged = [&](int node, int o) {
        double f[NRF];
#pragma unroll
        for (int k = 0; k < NRF; ++k) f[k] = rec[(Rot::field(k, o) * NN + node) * M + el];
        return EQ::from_rec(f, 0.0, 0.0, P);
    };

    double al[N][NV];
    int base = 0, s = 1;
    if (!faces) {
        // ---- volume terms of direction grp -----------------------------------
        const int o = grp;
        s = o == 0 ? 1 : (o == 1 ? N : N * N);
        base = o == 0 ? line_base<DIM, N>(line, 0) : (o == 1 ? line_base<DIM, N>(line, 1) : line_base<DIM, N>(line, 2));
        double alpha = 0.0, dg = 1.0;
        bool blended = false;
        if constexpr (VOL == VI_HG) {
            alpha = a.alpha_raw[ec];
            if (kc.smooth) {
#pragma unroll
                for (int f = 0; f < 2 * DIM; ++f) {
                    if (EXT && nb[f] < 0) {
                        if (nb[f] == -1) continue;  // boundary: no neighbour
                        const int32_t* mn = in_global(kc.mnb) + (int64_t)(-2 - nb[f]) * kc.mK;
                        for (int k = 0; k < kc.mK; ++k)
                            if (mn[k] >= 0) alpha = dmax(alpha, 0.5 * a.alpha_raw[mn[k]]);
                        continue;
                    }
                    alpha = dmax(alpha, 0.5 * a.alpha_raw[nb[f]]);
                }
            }
            blended = !(fabs(alpha) <= kc.atol);
            dg = blended ? 1.0 - alpha : 1.0;
        }
        Node nd[N];
#pragma unroll
        for (int p = 0; p < N; ++p) nd[p] = staged(base + p * s, o);
#pragma unroll
        for (int p = 0; p < N; ++p)
#pragma unroll
            for (int v = 0; v < NV; ++v) al[p][v] = 0.0;
        // the series means of every pair (branch free); a wave in which some
        // line has a jump of more than a third then does its volume terms over
        // again, one pair per turn with its checks: its nodes from LDS, its
        // flux added to all nodes, with weight zero where it does not belong
        // (registers are not indexed dynamically)
        bool near = true;
        if constexpr (LF && VF_LOGS) near = __builtin_amdgcn_ballot_w64(!EQ::template near_line<N>(nd)) == 0;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = i + 1; j < N; ++j) {
                double f[NV];
                node_flux<EQ, VF, TW, MEANS_NEAR, double, double>(nd[i], nullptr, nd[j], nullptr, 0, P, f);
                const double fa = VOL == VI_HG ? dg * kc.Ds[i * N + j] : kc.Ds[i * N + j];
                const double fb = VOL == VI_HG ? dg * kc.Ds[j * N + i] : kc.Ds[j * N + i];
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    al[i][v] += fa * f[v];
                    al[j][v] += fb * f[v];
                }
            }
        if (LF && VF_LOGS && !near) {
#pragma unroll
            for (int p = 0; p < N; ++p)
#pragma unroll
                for (int v = 0; v < NV; ++v) al[p][v] = 0.0;
#pragma unroll 1
            for (int i = 0; i + 1 < N; ++i)
#pragma unroll 1
                for (int j = i + 1; j < N; ++j) {
                    double f[NV];
                    node_flux<EQ, VF, TW, MEANS_ANY, double, double>(staged(base + i * s, o), nullptr,
                                                                     staged(base + j * s, o), nullptr, 0, P, f);
                    const double fa = dg * kc.Ds[i * N + j], fb = dg * kc.Ds[j * N + i];
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        const double w = p == i ? fa : (p == j ? fb : 0.0);
#pragma unroll
                        for (int v = 0; v < NV; ++v) al[p][v] += w * f[v];
                    }
                }
            // (read again, so that they hold no registers above)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int p = 0; p < N; ++p) nd[p] = staged(base + p * s, o);
        }
        if constexpr (EQ::NONCONS) line_noncons<N>(nd, kc.Ds, (TW ? 1.0 : 0.5) * dg, al);
        if (VOL == VI_HG && blended) {
#pragma unroll
            for (int p = 0; p + 1 < N; ++p) {
                double F[NV], ul[NV], ur[NV];
                if constexpr (flux_reads_cons(TW, FVF)) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        ul[v] = nd[p].cons(v);
                        ur[v] = nd[p + 1].cons(v);
                    }
                }
                node_flux<EQ, FVF, TW, MEANS_ANY, double, double>(nd[p], ul, nd[p + 1], ur, 0, P, F);
                const double wl = alpha * kc.invw[p], wr = alpha * kc.invw[p + 1];
                if constexpr (EQ::NONCONS) {
                    // the left node takes f + nc(u_l, u_r)/2, the right f + nc(u_r, u_l)/2
                    constexpr double h = TW ? 1.0 : 0.5;
                    double ncl[NV], ncr[NV];
                    EQ::template noncons<FVF>(nd[p], nd[p + 1], 0, P, ncl);
                    EQ::template noncons<FVF>(nd[p + 1], nd[p], 0, P, ncr);
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        al[p][v] += wl * (F[v] + h * ncl[v]);
                        al[p + 1][v] -= wr * (F[v] + h * ncr[v]);
                    }
                } else {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        al[p][v] += wl * F[v];
                        al[p + 1][v] -= wr * F[v];
                    }
                }
            }
        }
        if (grp == 0) {
#pragma unroll
            for (int p = 0; p < N; ++p)
#pragma unroll
                for (int v = 0; v < NV; ++v) acc[(Rot::variable(v, 0) * NN + base + p * s) * M + el] = al[p][v];
        }
    } else {
        // ---- interface fluxes of every direction -------------------------------
#pragma unroll 1
        for (int o = 0; o < DIM; ++o) {
            const int so = o == 0 ? 1 : (o == 1 ? N : N * N);
            const int bo = o == 0 ? line_base<DIM, N>(line, 0) : (o == 1 ? line_base<DIM, N>(line, 1) : line_base<DIM, N>(line, 2));
            double mc[NV], pc[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                mc[v] = um[v];
                pc[v] = up[v];
            }
            if (o + 1 < DIM) load_faces(o + 1, um, up);
            if constexpr (EXT) {
                int32_t nm = nb[0], np = nb[1];
#pragma unroll
                for (int f = 1; f < DIM; ++f) {
                    nm = o == f ? nb[2 * f] : nm;
                    np = o == f ? nb[2 * f + 1] : np;
                }
                if (kc.bc) {
                    // outflow and slip walls read the inner state (mc, pc hold
                    // it: this element's own face node on the other end is not
                    // it, so it is read here)
                    auto inner = [&](int node, double* x) {
#pragma unroll
                        for (int v = 0; v < NV; ++v) x[v] = U[soa(Rot::variable(v, o), node, ec, slab, E32)];
                    };
                    auto boundary = [&](int face, int node, double* x) {
                        if ((kc.outflow >> face) & 1) {
                            inner(node, x);
                        } else if (kc.bc == TRIXI_HIP_BC_SLIP_WALL) {
                            inner(node, x);
                            x[1] = -x[1];
                        } else {
                            double b[NV];
                            boundary_state<DIM, NN, NV, double>(a, kc, ec, node, tnow, b);
#pragma unroll
                            for (int v = 0; v < NV; ++v) {
                                const int w = Rot::variable(v, o);
#pragma unroll
                                for (int q = 0; q < NV; ++q)
                                    if (q == w) x[v] = b[q];
                            }
                        }
                    };
                    if (nm == -1) boundary(2 * o, bo, mc);
                    if (np == -1) boundary(2 * o + 1, bo + (N - 1) * so, pc);
                }
            }
            // one end after the other (fewer registers)
            auto face = [&](bool minus, double* uc, double* f) {
                const Node own = staged(minus ? bo : bo + (N - 1) * so, o);
                const Node nbn = EQ::template node<double, false, double>(uc, P);
                double uo[NV];
                if constexpr (flux_reads_cons(TW, SF)) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) uo[v] = own.cons(v);
                }
                if (minus)  // this element is "right"
                    node_flux<EQ, SF, TW, MEANS_ANY, double, double>(nbn, uc, own, uo, 0, P, f);
                else
                    node_flux<EQ, SF, TW, MEANS_ANY, double, double>(own, uo, nbn, uc, 0, P, f);
                if constexpr (EQ::NONCONS) {
                    constexpr double h = TW ? 1.0 : 0.5;
                    double nc[NV];
                    EQ::template noncons<SF>(own, nbn, 0, P, nc);
#pragma unroll
                    for (int v = 0; v < NV; ++v) f[v] += h * nc[v];
                }
            };
            double fm[NV], fp[NV];
            face(true, mc, fm);
            __builtin_amdgcn_sched_barrier(0);
            face(false, pc, fp);
            if constexpr (EXT) {
                // mortar faces: the face node of this line is `line`
                int32_t nm = nb[0], np = nb[1];
#pragma unroll
                for (int f = 1; f < DIM; ++f) {
                    nm = o == f ? nb[2 * f] : nm;
                    np = o == f ? nb[2 * f + 1] : np;
                }
                constexpr double h = TW ? 2.0 : 1.0;
                if (nm <= -2) {
                    const double* mf = in_global(kc.mflux) + ((int64_t)(-2 - nm) * NL + line) * NV;
#pragma unroll
                    for (int v = 0; v < NV; ++v) fm[v] = h * mf[Rot::variable(v, o)];
                }
                if (np <= -2) {
                    const double* mf = in_global(kc.mflux) + ((int64_t)(-2 - np) * NL + line) * NV;
#pragma unroll
                    for (int v = 0; v < NV; ++v) fp[v] = h * mf[Rot::variable(v, o)];
                }
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int w = Rot::variable(v, o);
                fcs[(((2 * o) * NL + line) * NV + w) * M + el] = -kc.lhat_m * fm[v];
                fcs[(((2 * o + 1) * NL + line) * NV + w) * M + el] = kc.lhat_p * fp[v];
            }
        }
    }

    // the lane index anew: its uses below would otherwise keep the node pass's
    // addresses in registers through the fluxes
    int tid2 = tid;
    asm volatile("" : "+v"(tid2));

    // the element's scale and dt, and u and k of the register update, requested
    // before the sums meet (a lane's nodes of the final pass are of one element:
    // NT is a multiple of M)
    static_assert(NT % M == 0, "a lane's nodes belong to one element");
    const double invj = a.invJ[e0 + tid2 % M < E ? e0 + tid2 % M : E - 1];
    double t_dt = 0.0;
    if (RK) t_dt = a.time[1];
    double uu[RK ? NIT : 1][NV], kk[RK ? NIT : 1][NV];
    const double* __restrict__ K = static_cast<const double*>(a.k);
    if constexpr (RK) {
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            int q = tid2 + it * NT;
            if ((it + 1) * NT > NN * M && q >= NN * M) q = NN * M - 1;
            const int64_t ee = e0 + q % M < E ? e0 + q % M : E - 1;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int64_t g = soa(v, q / M, ee, slab, E32);
                uu[it][v] = U[g];
                kk[it][v] = a.rk_first ? 0.0 : K[g];
            }
        }
    }
    __syncthreads();
    // direction 1 into the records' place, direction 2 added to direction 0
    if (grp == 1) {
#pragma unroll
        for (int p = 0; p < N; ++p)
#pragma unroll
            for (int v = 0; v < NV; ++v) rec[(Rot::variable(v, 1) * NN + base + p * s) * M + el] = al[p][v];
    }
    if (DIM > 2 && grp == 2) {
#pragma unroll
        for (int p = 0; p < N; ++p)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[(Rot::variable(v, 2) * NN + base + p * s) * M + el] += al[p][v];
    }
    __syncthreads();

    // ---- final pass: the node's sum, -1/J, sources, du or the register update --
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const int q = tid2 + it * NT;
        if ((it + 1) * NT > NN * M && q >= NN * M) continue;
        const int c = q % M, n = q / M;
        const int64_t e = e0 + c;
        if (e >= E) continue;
        double t[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) t[v] = acc[v * NN * M + q] + rec[v * NN * M + q];
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
        const double fac = (TW ? -0.5 : -1.0) * invj;
        double sv[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) sv[v] = 0.0;
        if (EXT && kc.src) source_at<DIM, NN, NV>(a, kc, e, n, tnow, sv);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t g = soa(v, n, e, slab, E32);
            const double val = t[v] * fac + sv[v];
            if constexpr (!RK) {
                static_cast<double*>(a.du)[g] = val;
            } else {
                const double kn = a.rk_first ? t_dt * val : a.rk_a * kk[it][v] + t_dt * val;
                static_cast<double*>(a.k)[g] = kn;
                static_cast<double*>(a.u_out)[g] = uu[it][v] + a.rk_b * kn;
            }
        }
    }
}

}  // namespace trixi_hip
