#pragma once
// One TR of a pSSFP isochromat as an affine map that depends on the TR's flip
// angle alone (pssfp_map.hip; the recursion itself is pssfp_common.h's).
//
// From the echo of TR n - 1 to the echo of TR n an isochromat goes through
// P E(rf_n) P: precession and relaxation over dt_pr (P), the RF pulse with
// its nRF sub-steps (E), and P again.  That is s' = B s + c with twelve
// numbers (B, c) that depend on the isochromat (T1, T2, B1, B0, z) and on
// rf_n, and on nothing else.  Write rf_n = theta e^{i phi}: the phase turns
// the rotation axes about z, E(rf) = Rz(-phi) E(theta) Rz(phi), and P commutes
// with Rz, so only the real amplitude theta is left.  E is a product of
// matrix exponentials that are linear in theta, so every entry is an entire
// function of theta, of exponential type L = max|rf| sum_k |g_k| B1 (the
// largest flip angle a pulse could reach), and E(-theta) = Rz(pi) E(theta)
// Rz(pi): Bxx, Bxy, Byx, Byy, Bzz, cz are even in theta, the other six odd.
// With theta in units of the train's largest amplitude and x = theta^2, each
// entry (odd ones over theta) is a polynomial in x on [0, 1] through MAP_NODES
// Chebyshev points.  Interpolation at n points in x leaves at most
// 2 (L/2)^(2n) / (2n)! of an even entry: 2e-12 at MAP_MAX_TYPE and n = 8; on
// the sinc-Gaussian pulse below 1e-14 up to 85 degrees (the bound supposes a
// pulse without sign changes).  Trains beyond MAP_MAX_TYPE take the sub-steps
// in every TR (pssfp_iso).

#include "compas/device/common.h"
#include "compas/device/pssfp_common.h"

namespace compas {
namespace kernels {

constexpr int MAP_NODES = 8;
constexpr double MAP_MAX_TYPE = 2.42;  // 2 (L/2)^16 / 16! <= 2e-12

// Chebyshev points (1 + cos((2 j + 1) pi / 16)) / 2 in Leja order (each the
// farthest, by product of distances, from those before it: the order in which
// Newton's form is stable), and their square roots.
constexpr double MAP_X[MAP_NODES] = {0.9903926402016152,  0.009607359798384785, 0.4024548389919359,  0.7777851165098011,
                                     0.22221488349019902, 0.9157348061512727,   0.08426519384872733, 0.5975451610080642};
constexpr double MAP_SQRT_X[MAP_NODES] = {0.9951847266721969, 0.09801714032956077, 0.6343932841636455,
                                          0.8819212643483549, 0.4713967368259978, 0.9569403357322088,
                                          0.29028467725446233, 0.773010453362737};

// Entries of a map: the first six even in theta, the last six odd
enum MapEntry : int { MXX, MXY, MYX, MYY, MZZ, MCZ, MXZ, MYZ, MZX, MZY, MCX, MCY, MAP_ENTRIES };

// Row n of a train's table: theta_n (in units of the largest amplitude), x_n -
// MAP_X[j] for j < MAP_NODES - 1, then cos and sin of phi_n - phi_{n-1}, and of
// phi_n.  Row -1 (the header, first in memory) holds the largest amplitude,
// whether the maps serve the train (1 or 0) and whether any phi_n is not zero.
constexpr int MAP_ROW = 16;
constexpr int MAP_PHASE = MAP_NODES;  // first of the four phase entries

struct PssfpMapArgs {
    PssfpArgs a;
    const double* train;  // [1 + nTR][MAP_ROW]
    // several slice-position groups: an FP64 plane of each, so that the sum is
    // rounded once (FP32 planes after the first: 3.0e-8 instead of 2.5e-8 on the
    // tangents of 35 positions in three groups).  Or, in the same memory, the FP32
    // planes of the sub-step form's groups after the first
    cfloat* partial;
    int nv_block;         // voxels of a workgroup
    int nz_group;         // slice positions of a group (nv_block nz_group <= 256)
    int vblocks, groups;  // ceil(nv / nv_block), ceil(nz / nz_group)
    int direct_zpl, direct_groups;  // slice positions per lane and groups of the sub-step form
};

// rotation_series with its constants held in scalar registers: an FMA whose
// addend is a literal would first move it into a vector register, two more
// instructions for each of the ten.
struct SeriesConst {
    double a[5], b[5];
    __device__ SeriesConst() :
        a {-1.0 / 39916800.0, 1.0 / 362880.0, -1.0 / 5040.0, 1.0 / 120.0, -1.0 / 6.0},
        b {-1.0 / 479001600.0, 1.0 / 3628800.0, -1.0 / 40320.0, 1.0 / 720.0, -1.0 / 24.0} {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            asm("" : "+s"(a[i]));
            asm("" : "+s"(b[i]));
        }
    }
    __device__ void operator()(double u, double& s1, double& s2) const {
        s1 = fma(u, a[0], a[1]);
        s2 = fma(u, b[0], b[1]);
#pragma unroll
        for (int i = 2; i < 5; i++) {
            s1 = fma(u, s1, a[i]);
            s2 = fma(u, s2, b[i]);
        }
        s1 = fma(u, s1, 1.0);
        s2 = fma(u, s2, 0.5);
    }
};

// M = relaxation x rotation of one RF sub-step about (ax, ay, az): Rodrigues'
// matrix c I + s1 [a]x + s2 a a^T, rows scaled by E2, E2, E1.
__device__ inline void substep_matrix(
    const SeriesConst& series, double ax, double ay, double az, double E1, double E2, double (&M)[9]) {
    const double u = fma(ax, ax, fma(ay, ay, az * az));
    double s1, s2;
    if (!__any(u > SERIES_LIMIT)) {
        series(u, s1, s2);
    } else {
        rotation_any(u, s1, s2);
    }
    const double c = fma(-u, s2, 1.0);
    const double tx = s2 * ax, ty = s2 * ay;
    const double sx = s1 * ax, sy = s1 * ay, sz = s1 * az;
    const double xy = tx * ay, xz = tx * az, yz = ty * az;
    M[0] = fma(tx, ax, c) * E2;
    M[1] = (xy - sz) * E2;
    M[2] = (xz + sy) * E2;
    M[3] = (xy + sz) * E2;
    M[4] = fma(ty, ay, c) * E2;
    M[5] = (yz - sx) * E2;
    M[6] = (xz - sy) * E1;
    M[7] = (yz + sx) * E1;
    M[8] = fma(s2 * az, az, c) * E1;
}

__device__ inline void apply3(const double (&M)[9], Vec3d& m) {
    const double x = fma(M[0], m.x, fma(M[1], m.y, M[2] * m.z));
    const double y = fma(M[3], m.x, fma(M[4], m.y, M[5] * m.z));
    const double z = fma(M[6], m.x, fma(M[7], m.y, M[8] * m.z));
    m = {x, y, z};
}

// What a lane holds of its isochromat besides its map
struct IsoConst {
    double B1, az;
    double E1, E2, R1;      // one RF sub-step
    double pc, ps, P1, Q1;  // dt_pr: E2 cos, E2 sin, E1, 1 - E1
};

__device__ inline void precess(const IsoConst& k, Vec3d& m, double regrow) {
    const double x = fma(k.pc, m.x, -k.ps * m.y), y = fma(k.pc, m.y, k.ps * m.x);
    m = {x, y, fma(k.P1, m.z, regrow)};
}

}  // namespace kernels
}  // namespace compas
