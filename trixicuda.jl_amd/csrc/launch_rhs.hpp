// launch_rhs.hpp -- which form of the rhs! kernel a configuration runs.
#pragma once

#include "rhs_group_kernel.hpp"

namespace trixi_hip {

// Shapes of the lane-group form: FP64 flux differencing and shock capturing in
// 2D and 3D for the equations with a rotation, whole waves per group.
template <class EQ>
struct HasRotation : std::false_type {};
template <int DIM>
struct HasRotation<Euler<DIM>> : std::true_type {};
template <>
struct HasRotation<GlmMhd> : std::true_type {};

#ifndef TRIXI_HIP_GROUP_LDS_KIB
#define TRIXI_HIP_GROUP_LDS_KIB 78
#endif
// Elements per workgroup: the most (a power of two) whose LDS leaves room for
// two workgroups per compute unit, at most 16.
template <int DIM, int N, int NV, int NRF>
constexpr int group_elems() {
    constexpr int NL = cpow(N, DIM - 1), NN = cpow(N, DIM);
    int m = 16;
    while (m > 1 && m * 8 * (NRF * NN + NV * NN + DIM * 2 * NL * NV) > TRIXI_HIP_GROUP_LDS_KIB * 1024) m /= 2;
    return m;
}
// element lines from which lines_when_large forms take lines
#ifndef TRIXI_HIP_GROUP_LINE_LANES
#define TRIXI_HIP_GROUP_LINE_LANES 65536
#endif
#ifndef TRIXI_HIP_GROUP_WAVES2D
#define TRIXI_HIP_GROUP_WAVES2D 3
#endif
template <int DIM, int N, class EQ, int VOL, typename R>
constexpr bool group_eligible() {
    return std::is_same<R, double>::value && DIM > 1 && VOL != VI_WEAK && HasRotation<EQ>::value &&
           (group_elems<DIM, N, EQ::NV, EQ::NRF>() * cpow(N, DIM - 1)) % 64 == 0 &&
           group_threads<DIM, N, group_elems<DIM, N, EQ::NV, EQ::NRF>()>() <= 1024;
}

// rhs! in 2D, and of Euler's shock capturing without logarithmic means in 3D, takes
// the line form on meshes that fill the GPU with it (a wave per SIMD and direction):
// its rows are as wide there, and it has no group that the others wait for.  rhs! in
// us, lane groups / lines: 2D at 16384 elements GLM-MHD 17.6 / 15.2, shock capturing
// 16.0 / 15.2; at 65536 Euler 21.0 / 18.8, without logarithms 19.6 / 15.7, shock
// capturing 44.8 / 42.8; 3D shock capturing without logarithms at 4096 32.9 / 31.4, at
// 32768 173 / 165.  Below, lane groups have more lanes (2D GLM-MHD at 4096 8.3 / 12).
// The RK stages, which read u and k besides, gain from lane groups everywhere (2D
// GLM-MHD at 65536 94 / 156), and so do 3D flux differencing (Euler at 32768 80 / 84),
// 3D shock capturing with logarithms (at 4096 33.0 / 33.8, at 32768 176 / 187) and 3D
// GLM-MHD (shock capturing at 4096 53.5 / 55.0).
template <int DIM, class EQ, int VOL, int VF, bool RK, bool EXT>
constexpr bool lines_when_large() {
    return !RK && !EXT && (DIM == 2 || (VOL == VI_HG && !EQ::NONCONS && !flux_needs_logs(VF)));
}

// Launch helper used by the instantiation units: the node-parallel form for
// small periodic conforming meshes (RhsArgs::np), the lane-group form where it
// is built, the line form otherwise.
template <int DIM, int N, class EQ, int VOL, int VF, int SF, int FVF, typename R, int M, bool RK, bool EXT = false,
          typename L = double, typename S = double>
hipError_t launch_rhs(const RhsArgs& a, hipStream_t stream) {
    auto consts = [&]() -> RhsConstArg<R> {
        if constexpr (std::is_same<R, double>::value)
            return a.consts;
        else
            return *a.host_consts;
    };
    auto grid = [&](int m) {
        int64_t blocks = (a.E + m - 1) / m;
        if (a.nxcd > 1) blocks = (blocks + a.nxcd - 1) / a.nxcd * a.nxcd;
        return dim3((unsigned)blocks);
    };
    if constexpr (np_eligible<DIM, N, EQ::NV, VOL, EXT>()) {
        if (a.np) {
            constexpr int MN = np_elems<DIM, N>();
            hipLaunchKernelGGL((rhs_np_kernel<DIM, N, EQ, VOL, VF, SF, FVF, R, RK, L, S>), grid(MN),
                               dim3(MN * cpow(N, DIM) * DIM), 0, stream, a, consts());
            return hipGetLastError();
        }
    }
    // only the node-parallel form computes the next stage's blending factors
    if (a.alpha_next != nullptr) return hipErrorInvalidValue;
    if constexpr (group_eligible<DIM, N, EQ, VOL, R>()) {
        constexpr int ME = group_elems<DIM, N, EQ::NV, EQ::NRF>();
        // Half the elements and two waves per SIMD (256 registers) where four
        // waves spill: boundary and mortar faces, and shock capturing in 3D,
        // whose blended lines hold 60 registers too many (rhs! at 32768
        // elements 219 -> 180 us, three CFL steps 4360 -> 3320; with three
        // waves the same).  In 2D the tiles cannot be halved (whole waves), and
        // three waves hold boundary and mortar faces as well (65536 elements with
        // Dirichlet faces: rhs! 48.3 -> 37.0 us, RK stage 63.9 -> 51.4).
        constexpr bool HALF = (EXT || VOL == VI_HG) && DIM == 3;
        constexpr int MG = HALF && (ME / 2 * cpow(N, DIM - 1)) % 64 == 0 ? ME / 2 : ME;
        constexpr int W = EQ::NV > 5 || HALF ? 2 : (DIM == 3 ? 4 : TRIXI_HIP_GROUP_WAVES2D);
        constexpr bool LINES = lines_when_large<DIM, EQ, VOL, VF, RK, EXT>();
        if (!LINES || a.E * cpow(N, DIM - 1) < TRIXI_HIP_GROUP_LINE_LANES) {
            hipLaunchKernelGGL((rhs_group_kernel<DIM, N, EQ, VOL, VF, SF, FVF, MG, RK, EXT, W>), grid(MG),
                               dim3(group_threads<DIM, N, MG>()), 0, stream, a, a.consts);
            return hipGetLastError();
        }
    }
    if constexpr (!group_eligible<DIM, N, EQ, VOL, R>() || lines_when_large<DIM, EQ, VOL, VF, RK, EXT>()) {
        hipLaunchKernelGGL((rhs_kernel<DIM, N, EQ, VOL, VF, SF, FVF, R, M, RK, EXT, L, S>), grid(M),
                           dim3(rhs_threads<DIM, N, M, R, RK, EQ::NV>()), 0, stream, a, consts());
    }
    return hipGetLastError();
}

}  // namespace trixi_hip
