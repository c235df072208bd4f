// Tangent passes of the real-valued FISP recursion (compas/device/fisp_real.h).

#include <algorithm>

#include "compas/device/common.h"
#include "compas/device/fisp_common.h"
#include "compas/device/fisp_real.h"
#include "compas/internal.h"

namespace compas {
namespace kernels {

template<int SPL, int LPV, int MASK>
__global__ void __launch_bounds__(64) fisp_real_tangents(FispArgs a, FispPlanes out) {
    if (!fisp_real_train(a)) return;  // fisp_epg_tangents runs instead
    const int sub = (LPV > 1) ? int(threadIdx.x % LPV) : 0;
    const int voxel = (blockIdx.x * 64 + threadIdx.x) / LPV;
    if (voxel >= a.tissue.nvoxels) return;  // whole LPV groups leave together
    fisp_real_voxel<SPL, LPV, MASK>(a, out, voxel, sub);
}

}  // namespace kernels

namespace {

using namespace kernels;

using Launcher = void (*)(const FispArgs&, const FispPlanes&, unsigned, hipStream_t);

template<int SPL, int LPV, int MASK>
void launch(const FispArgs& a, const FispPlanes& out, unsigned blocks, hipStream_t s) {
    fisp_real_tangents<SPL, LPV, MASK><<<blocks, 64, 0, s>>>(a, out);
}

// Two or eight lanes per voxel, up to sixteen states in each
template<int MASK, int LPV, int SPL = 1>
Launcher find(int spl) {
    if (spl == SPL) return &launch<SPL, LPV, MASK>;
    if constexpr (SPL < 16) return find<MASK, LPV, SPL + 1>(spl);
    return nullptr;
}

template<int MASK>
Launcher find(int lpv, int spl) {
    return lpv == 2 ? find<MASK, 2>(spl) : find<MASK, 8>(spl);
}

// Lanes per voxel: the lower modelled time of a TR.  nv: vectors carried (the
// state and its tangents).  A wave alone on its SIMD is bound by its chain of
// operations, several by the instructions issued; both grow with the states
// per lane, and in proportion to a part that every lane repeats.  Constants
// (in us per TR) fitted to the T1 + T2 pass: 50176 voxels x 25 states 1.14 in
// two lanes, 1.64 in eight; 1000 voxels 1.05 and 0.50; 4096 x 16 0.69 and 0.45.
int choose_lanes(int N, int voxels, int simds, int nv) {
    if (N > 32) return 8;
    double best = 1e300;
    int best_l = 8;
    for (int l : {2, 8}) {
        const int s = (N + l - 1) / l;
        const double waves = double(voxels) * l / 64.0 / simds;
        const double alone = 0.08 + 0.075 * nv + 0.018 * nv * s;
        const double shared = 0.3 + waves * (0.015 + 0.02 * nv + 0.0133 * nv * s);
        if (std::max(alone, shared) < best) {
            best = std::max(alone, shared);
            best_l = l;
        }
    }
    return best_l;
}

}  // namespace

void launch_fisp_real_tangents(const CompasContext& ctx, const FispArgs& a, int mask, const FispPlanes& planes) {
    FispPlanes out = planes;
    const int fields = mask & ~TM_ECHO;
    const bool single = fields == TM_T1 || fields == TM_T2 || fields == TM_B1 || fields == TM_B0;
    if (!single && !(mask & TM_ECHO)) {  // the kernels of several fields have a place for the echoes
        for (int k = 4; k > 0; k--) out.p[k] = out.p[k - 1];
        out.p[0] = nullptr;
    }
    const int nv = fields == TM_B0 ? 1 : single ? 2 : fields == (TM_T1 | TM_T2) ? 3 : 4;
    const int lpv = choose_lanes(a.N, a.tissue.nvoxels, simd_count(ctx.device()), nv);
    const int spl = (a.N + lpv - 1) / lpv;
    Launcher fn = nullptr;
    switch (fields) {
        case TM_T1: fn = find<TM_T1>(lpv, spl); break;
        case TM_T2: fn = find<TM_T2>(lpv, spl); break;
        case TM_B1: fn = find<TM_B1>(lpv, spl); break;
        case TM_B0: fn = find<TM_B0>(lpv, spl); break;
        case TM_T1 | TM_T2: fn = find<TM_T1 | TM_T2 | TM_ECHO>(lpv, spl); break;
        case TM_T1 | TM_T2 | TM_B1 | TM_B0: fn = find<TM_T1 | TM_T2 | TM_B1 | TM_B0 | TM_ECHO>(lpv, spl); break;
        default: break;
    }
    COMPAS_CHECK(fn != nullptr);
    fn(a, out, dev::div_ceil(int64_t(a.tissue.nvoxels) * lpv, 64), ctx.stream());
    check_launch("fisp_real_tangents");
}

}  // namespace compas
