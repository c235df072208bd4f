#pragma once
// Per-voxel constants and phasors of the spiral sample factor
//   E_rv^s = exp(s (-dt / T2_v + i (dk_r . x_v + 2 pi dt B0_v)))
// (spiral_view.cuh:59-73) shared by the two-level spiral kernels.

#include "compas/device/common.h"

namespace compas {
namespace kernels {

// One voxel: x, y, dt B0 in turns, and the decay exponent per sample, base 2
struct alignas(16) SpiralVoxel {
    double turns;
    float x, y;
    float decay;
    float T2;
    float pad[2];
};

// Written beside a kernel that runs before the products anyway: a launch of its
// own made the smallest calls slower than the products gained
__device__ inline SpiralVoxel spiral_voxel(const dev::TissueView& t, float dt, int v) {
    SpiralVoxel o {};
    o.turns = double(dt) * double(t.B0(v));
    o.x = t.x(v);
    o.y = t.y(v);
    o.T2 = t.T2(v);
    o.decay = float(-1.4426950408889634 * double(dt) / double(o.T2));  // log2(e)
    return o;
}

// Turns per sample of a voxel; dkx, dky: delta_k / 2 pi
__device__ __forceinline__ double spiral_turns(const SpiralVoxel& v, double dkx, double dky) {
    return fma(dkx, double(v.x), fma(dky, double(v.y), v.turns));
}

// 2^(log2_mag) e^{2 pi i turns}: the phase is reduced to half a turn in FP64.
// With the hardware's sine and cosine of a phase in turns and its base-2
// exponential the result is within 7.2e-8 (RMS, relative; 2.2e-7 at most): more
// than sincos_reduced and expf leave (5.9e-8), at a third of the instructions.
// The factor E^s that two levels make of it passes through fewer products than a
// sequence over all samples: RMS over 512 samples 6.6e-7 in the sums (a sequence
// of 32 steps of sixteen samples by sincos_reduced and expf 1.1e-6) and 5.3e-7 in
// J^H.y (5.5e-7).
__device__ __forceinline__ cfloat spiral_phasor(float log2_mag, double turns) {
    const float f = float(turns - rint(turns));
    const float m = __builtin_amdgcn_exp2f(log2_mag);
    return {m * __builtin_amdgcn_cosf(f), m * __builtin_amdgcn_sinf(f)};
}

}  // namespace kernels
}  // namespace compas
