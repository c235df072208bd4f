#pragma once
// The per-call kernel of the complex FISP recursion and its launchers
// (fisp_lanes.hip: one lane per voxel; fisp_lanes_2.hip: two; fisp_lanes_n.hip:
// four and eight).

#include "compas/device/fisp_epg.h"
#include "compas/device/fisp_real.h"

namespace compas {

using FispLauncher = void (*)(const kernels::FispArgs&, unsigned, hipStream_t);

// nullptr where there is no kernel of this layout
FispLauncher fisp_epg_launcher_1(int spl);
FispLauncher fisp_epg_launcher_2(int spl);
FispLauncher fisp_epg_launcher_n(int lpv, int spl);
inline FispLauncher fisp_epg_launcher(int lpv, int spl) {
    return lpv == 1 ? fisp_epg_launcher_1(spl) : lpv == 2 ? fisp_epg_launcher_2(spl) : fisp_epg_launcher_n(lpv, spl);
}

namespace kernels {

template<int SPL, int LPV>
__global__ void __launch_bounds__(64) fisp_epg(FispArgs a) {
    const int sub = (LPV > 1) ? int(threadIdx.x % LPV) : 0;
    const int voxel = (blockIdx.x * 64 + threadIdx.x) / LPV;
    if (fisp_real_train(a)) return;  // fisp_real runs instead
    if (voxel >= a.tissue.nvoxels) return;  // whole LPV groups leave together
    fisp_epg_voxel<SPL, LPV>(a, voxel, sub);
}

}  // namespace kernels

template<int SPL, int LPV>
void launch_fisp_epg_kernel(const kernels::FispArgs& a, unsigned blocks, hipStream_t stream) {
    kernels::fisp_epg<SPL, LPV><<<blocks, 64, 0, stream>>>(a);
}

template<int LPV, int SPL, int MAX>
FispLauncher find_fisp_epg(int spl) {
    if (spl == SPL) return &launch_fisp_epg_kernel<SPL, LPV>;
    if constexpr (SPL < MAX) return find_fisp_epg<LPV, SPL + 1, MAX>(spl);
    return nullptr;
}

}  // namespace compas
