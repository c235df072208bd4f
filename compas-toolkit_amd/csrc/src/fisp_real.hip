// Launches of the real-valued FISP recursion and its tangents
// (compas/device/fisp_real.h): trains whose RF pulses are real.  The complex
// form (fisp.hip, fisp_tangent.hip) is launched beside it for the others.

#include <algorithm>
#include <cstdlib>

#include "compas/device/common.h"
#include "compas/device/fisp_common.h"
#include "compas/device/fisp_real.h"
#include "compas/internal.h"

namespace compas {
namespace kernels {

template<int SPL, int LPV, int MASK>
__global__ void __launch_bounds__(64) fisp_real(FispArgs a, FispPlanes out) {
    if (!fisp_real_train(a)) return;  // fisp_epg or fisp_epg_tangents runs instead
    const int sub = (LPV > 1) ? int(threadIdx.x % LPV) : 0;
    const int voxel = (blockIdx.x * 64 + threadIdx.x) / LPV;
    if (voxel >= a.tissue.nvoxels) return;  // whole LPV groups leave together
    fisp_real_voxel<SPL, LPV, MASK>(a, out, voxel, sub);
}

}  // namespace kernels

namespace {

using namespace kernels;

using RealLauncher = void (*)(const FispArgs&, const FispPlanes&, unsigned, hipStream_t);

template<int SPL, int LPV, int MASK>
void launch(const FispArgs& a, const FispPlanes& out, unsigned blocks, hipStream_t s) {
    fisp_real<SPL, LPV, MASK><<<blocks, 64, 0, s>>>(a, out);
}

template<int LPV, int SPL, int MAX>
RealLauncher find(int spl) {
    if (spl == SPL) return &launch<SPL, LPV, TM_ECHO>;
    if constexpr (SPL < MAX) return find<LPV, SPL + 1, MAX>(spl);
    return nullptr;
}

RealLauncher find(int lpv, int spl) {
    switch (lpv) {
        case 1: return find<1, 1, 32>(spl);
        case 2: return find<2, 1, 16>(spl);
        case 4: return find<4, 1, 16>(spl);
        default: return find<8, 1, 16>(spl);
    }
}

// Lanes per voxel: the lowest modelled time of a TR.  A wave alone on its SIMD
// is bound by its chain of operations, several by the instructions issued.
// Constants (in us per TR) fitted to, in 1, 2, 4 and 8 lanes: 50176 voxels x
// 25 states 0.43, 0.40, 0.48, 0.60; 200000 x 25 1.01, 1.23, 1.47, 2.07;
// 20000 x 25 0.43, 0.34, 0.30, 0.31; 4096 x 16 0.32, 0.28, 0.23, 0.19.
int choose_lanes(int N, int nvoxels, int simds) {
    if (const char* e = std::getenv("COMPAS_FISP_LPV")) {  // layout override
        const int l = std::atoi(e);
        if ((l == 1 && N <= 32) || ((l == 2 || l == 4 || l == 8) && (N + l - 1) / l <= 16)) return l;
    }
    int best_l = 8;
    double best = 1e300;
    for (int l : {1, 2, 4, 8}) {
        const int s = (N + l - 1) / l;
        if (s > (l == 1 ? 32 : 16)) continue;
        const double waves = double(nvoxels) * l / 64.0 / simds;
        const double cost = std::max(0.155 + 0.0108 * s, 0.15 + waves * (0.05 + 0.0095 * s));
        if (cost < best) {
            best = cost;
            best_l = l;
        }
    }
    return best_l;
}

}  // namespace

void launch_fisp_real(const CompasContext& ctx, const FispArgs& a, int mask, const FispPlanes& out) {
    if (!(a.wait_spoiling || a.inversion || a.repetitions == 1)) return;  // fisp_real_train
    if (mask != TM_ECHO) {
        launch_fisp_real_tangents(ctx, a, mask, out);
        return;
    }
    const int lpv = choose_lanes(a.N, a.tissue.nvoxels, simd_count(ctx.device()));
    const RealLauncher fn = find(lpv, (a.N + lpv - 1) / lpv);
    COMPAS_CHECK(fn != nullptr);
    fn(a, out, dev::div_ceil(int64_t(a.tissue.nvoxels) * lpv, 64), ctx.stream());
    check_launch("fisp_real");
}

}  // namespace compas
