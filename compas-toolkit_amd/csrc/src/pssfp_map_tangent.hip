// Forward-mode derivatives of the pSSFP simulation by per-TR maps (gfx950).
//
// pssfp_map.h writes a TR of an isochromat as s' = B s + c with entries that are
// polynomials in the TR's flip angle.  With respect to a tissue parameter p the
// tangent obeys ds' = B ds + B_p s + c_p, and the entries of (B_p, c_p) are
// polynomials of the same kind and parity, so one pass evaluates two maps per
// TR where the sub-step form (pssfp_tangent.hip) takes every RF sub-step through
// the rotation and its derivative.
//
//   * pssfp_map_nodes: thread (isochromat, node) takes the four columns of the
//     pulse's affine map and their tangents through the sub-steps at the node's
//     flip angle; node MAP_NODES takes the state itself to the first echo.
//   * pssfp_map_tangents: 2 NF lanes per isochromat, NF <= 2 fields in a pass:
//     lane (field f, half h) holds the coefficients of its half of its field's
//     map, the row of x (h = 0) or y (h = 1) and its share of z's row: six
//     entries, 96 VGPRs.  The map of the state itself is shared by the two
//     fields, three entries to a lane.  Each half advances its own component of
//     the state and of the tangent; the halves swap components by DPP.
//   * The sum over slice positions as in pssfp_map.hip; a workgroup holds 64 or 128
//     isochromats, so there are several groups, with an FP64 plane each, from
//     about thirty positions on.
//
// What bounds it: FP64 issue.  All four fields and the echoes (two passes) at
// 3136 voxels x 280 TRs x 35 positions x 25 sub-steps take 1.7 ms (5.6 by
// sub-steps), 0.56 of them the nodes; at 50176 x 1120 83 ms (271), T1 + T2 at
// 3136 x 280 0.83 (4.3), B1 alone 0.82 (6.7).

#include <algorithm>
#include <vector>

#include "compas/device/common.h"
#include "compas/device/pssfp_common.h"
#include "compas/device/pssfp_map.h"
#include "compas/device/tangent_set.h"
#include "compas/internal.h"
#include "compas/pssfp_layout.h"

namespace compas {
namespace kernels {

constexpr int MAPT_CHUNK = 8;  // TRs summed over slice positions at a time

// v of the lane that the quad permutation names
template<int CONTROL>
__device__ __forceinline__ double quad(double v) {
    const int2 w = __builtin_bit_cast(int2, v);
    const int2 o = {__builtin_amdgcn_mov_dpp(w.x, CONTROL, 0xF, 0xF, true),
                    __builtin_amdgcn_mov_dpp(w.y, CONTROL, 0xF, 0xF, true)};
    return __builtin_bit_cast(double, o);
}

struct Mat3 {
    double a[9];
    __device__ Vec3d operator*(const Vec3d& v) const {
        return {fma(a[0], v.x, fma(a[1], v.y, a[2] * v.z)), fma(a[3], v.x, fma(a[4], v.y, a[5] * v.z)),
                fma(a[6], v.x, fma(a[7], v.y, a[8] * v.z))};
    }
};

// c I + [w]x + p a^T (p: s2 a)
__device__ inline Mat3 rotation_form(double c, Vec3d w, Vec3d p, Vec3d a) {
    return {{fma(p.x, a.x, c), fma(p.x, a.y, -w.z), fma(p.x, a.z, w.y), fma(p.y, a.x, w.z), fma(p.y, a.y, c),
             fma(p.y, a.z, -w.x), fma(p.z, a.x, -w.y), fma(p.z, a.y, w.x), fma(p.z, a.z, c)}};
}

// d/dp of c I + s1 [a]x + s2 a a^T along da
__device__ inline Mat3 rotation_derivative(
    Vec3d a, Vec3d da, double u, double s1, double s2, double s1p, double s2p) {
    const double du = 2.0 * fma(a.x, da.x, fma(a.y, da.y, a.z * da.z));
    const double dc = -fma(u, s2p, s2) * du, d1 = s1p * du, d2 = s2p * du;
    const Vec3d w = {fma(d1, a.x, s1 * da.x), fma(d1, a.y, s1 * da.y), fma(d1, a.z, s1 * da.z)};
    const Vec3d p = {fma(d2, a.x, s2 * da.x), fma(d2, a.y, s2 * da.y), fma(d2, a.z, s2 * da.z)};
    Mat3 m = rotation_form(dc, w, p, a);
    const Vec3d q = {s2 * a.x, s2 * a.y, s2 * a.z};
    m.a[0] = fma(q.x, da.x, m.a[0]);
    m.a[1] = fma(q.x, da.y, m.a[1]);
    m.a[2] = fma(q.x, da.z, m.a[2]);
    m.a[3] = fma(q.y, da.x, m.a[3]);
    m.a[4] = fma(q.y, da.y, m.a[4]);
    m.a[5] = fma(q.y, da.z, m.a[5]);
    m.a[6] = fma(q.z, da.x, m.a[6]);
    m.a[7] = fma(q.z, da.y, m.a[7]);
    m.a[8] = fma(q.z, da.z, m.a[8]);
    return m;
}

struct MapTangentArgs {
    PssfpMapArgs p;  // partial: NP planes of each group
    cfloat* out[3];  // output planes, in the order of TangentSet
    double* nodes;   // [1 + NT maps][MAP_NODES][MAP_ENTRIES][isos], then [3 + 3 NT][isos]
    int v0, nv;      // voxels of this launch
};

// The chunk's isochromat i: voxel v0 + i / nz, slice position i % nz
template<int MASK>
__global__ void __launch_bounds__(256, 2) pssfp_map_nodes(MapTangentArgs t) {
    using TS = TangentSet<MASK>;
    constexpr int NT = TS::nt;
    const PssfpArgs& a = t.p.a;
    __shared__ double2 grf[RF_CHUNK];
    const double* train = t.p.train;
    if (train[1] == 0.0) return;
    for (int i = threadIdx.x; i < a.nRF; i += 256) grf[i] = make_double2(double(a.gamma_dt_RF[i].re), double(a.gamma_dt_RF[i].im));
    __syncthreads();
    const int64_t isos = int64_t(t.nv) * a.nz;
    const int64_t iso = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int64_t at = min(iso, isos - 1);
    const int voxel = t.v0 + int(at / a.nz), node = blockIdx.y;
    const double zz = a.z[int(at % a.nz)];

    const double T1 = a.tissue.T1(voxel), T2 = a.tissue.T2(voxel), B1 = a.tissue.B1(voxel), B0 = a.tissue.B0(voxel);
    const double dt_ex = a.dt_ex, dt_pr = a.dt_pr, dt_inv = a.dt_inv;
    const double k1 = 1.0 / (T1 * T1), k2 = 1.0 / (T2 * T2);
    const double E1 = exp(-dt_ex / T1), E2 = exp(-dt_ex / T2), dE1 = dt_ex * k1 * E1, dE2 = dt_ex * k2 * E2;
    const double E1p = exp(-dt_pr / T1), E2p = exp(-dt_pr / T2), dE1p = dt_pr * k1 * E1p, dE2p = dt_pr * k2 * E2p;
    const double az = -(double(a.g_ex) * zz) - dt_ex * dev::TWO_PI * B0;
    const double daz = -dev::TWO_PI * dt_ex, dth = -dev::TWO_PI * dt_pr;

    // relaxation of one vector and its tangents; grow: with regrowth
    auto relax = [&](Vec3d& m, Vec3d (&d)[NT], double e1, double e2, double de1, double de2, bool grow) {
#pragma unroll
        for (int k = 0; k < NT; k++) {
            d[k].x *= e2;
            d[k].y *= e2;
            d[k].z *= e1;
            if (TS::t2 && k == TS::it2) {
                d[k].x = fma(m.x, de2, d[k].x);
                d[k].y = fma(m.y, de2, d[k].y);
            }
            if (TS::t1 && k == TS::it1) d[k].z = fma(grow ? m.z - 1.0 : m.z, de1, d[k].z);
        }
        m.x *= e2;
        m.y *= e2;
        m.z = grow ? fma(m.z, e1, 1.0 - e1) : m.z * e1;
    };
    auto precess_all = [&](Vec3d& m, Vec3d (&d)[NT], double c, double s, bool grow) {
        rotate_z(m, c, s);
#pragma unroll
        for (int k = 0; k < NT; k++) rotate_z(d[k], c, s);
        if constexpr (TS::b0) {
            d[TS::ib0].x = fma(-dth, m.y, d[TS::ib0].x);
            d[TS::ib0].y = fma(dth, m.x, d[TS::ib0].y);
        }
        relax(m, d, E1p, E2p, dE1p, dE2p, grow);
    };
    // the sub-steps of one pulse on NV vectors, the last of them with regrowth
    auto pulse_all = [&](auto& m, auto& d, auto count, double re, double im) {
        constexpr int NV = decltype(count)::value;
        const SeriesConst series;
        for (int i = 0; i < a.nRF; i++) {
            const double2 g = grf[i];
            const double zre = re * g.x - im * g.y, zim = re * g.y + im * g.x;
            const Vec3d ax = {zre * B1, -zim * B1, az};
            const double u = fma(ax.x, ax.x, fma(ax.y, ax.y, az * az));
            double s1, s2, s1p = 0.0, s2p = 0.0;
            if (!__any(u > SERIES_LIMIT)) {
                series(u, s1, s2);
            } else {
                rotation_any(u, s1, s2);
            }
            if constexpr (TS::axis) {
                // term-wise derivatives of the two series, one more term each; above
                // half a radian the closed forms
                if (!__any(u > SERIES_LIMIT_WIDE)) {
                    s1p = fma(u, -7.0 / 1307674368000.0, 6.0 / 6227020800.0);
                    s1p = fma(u, s1p, -5.0 / 39916800.0);
                    s1p = fma(u, s1p, 4.0 / 362880.0);
                    s1p = fma(u, s1p, -3.0 / 5040.0);
                    s1p = fma(u, s1p, 2.0 / 120.0);
                    s1p = fma(u, s1p, -1.0 / 6.0);
                    s2p = fma(u, -7.0 / 20922789888000.0, 6.0 / 87178291200.0);
                    s2p = fma(u, s2p, -5.0 / 479001600.0);
                    s2p = fma(u, s2p, 4.0 / 3628800.0);
                    s2p = fma(u, s2p, -3.0 / 40320.0);
                    s2p = fma(u, s2p, 2.0 / 720.0);
                    s2p = fma(u, s2p, -1.0 / 24.0);
                } else {
                    const double c = fma(-u, s2, 1.0), w = u > SERIES_LIMIT_WIDE ? u : 1.0;
                    s1p = (c - s1) / (2.0 * w);
                    s2p = (s1 - 2.0 * s2) / (2.0 * w);
                    if (u <= SERIES_LIMIT_WIDE) {
                        s1p = -1.0 / 6.0 + u * (2.0 / 120.0 + u * (-3.0 / 5040.0 + u * (4.0 / 362880.0 + u * (-5.0 / 39916800.0 + u * (6.0 / 6227020800.0 - u * (7.0 / 1307674368000.0))))));
                        s2p = -1.0 / 24.0 + u * (2.0 / 720.0 + u * (-3.0 / 40320.0 + u * (4.0 / 3628800.0 + u * (-5.0 / 479001600.0 + u * (6.0 / 87178291200.0 - u * (7.0 / 20922789888000.0))))));
                    }
                }
            }
            const double c = fma(-u, s2, 1.0);
            const Mat3 R = rotation_form(c, {s1 * ax.x, s1 * ax.y, s1 * ax.z}, {s2 * ax.x, s2 * ax.y, s2 * ax.z}, ax);
#pragma unroll
            for (int v = 0; v < NV; v++)
#pragma unroll
                for (int k = 0; k < NT; k++) d[v][k] = R * d[v][k];
            if constexpr (TS::b1) {
                const Mat3 Q = rotation_derivative(ax, {zre, -zim, 0.0}, u, s1, s2, s1p, s2p);
#pragma unroll
                for (int v = 0; v < NV; v++) {
                    const Vec3d x = Q * m[v];
                    Vec3d& y = d[v][TS::ib1];
                    y = {y.x + x.x, y.y + x.y, y.z + x.z};
                }
            }
            if constexpr (TS::b0) {
                const Mat3 Q = rotation_derivative(ax, {0.0, 0.0, daz}, u, s1, s2, s1p, s2p);
#pragma unroll
                for (int v = 0; v < NV; v++) {
                    const Vec3d x = Q * m[v];
                    Vec3d& y = d[v][TS::ib0];
                    y = {y.x + x.x, y.y + x.y, y.z + x.z};
                }
            }
#pragma unroll
            for (int v = 0; v < NV; v++) {
                m[v] = R * m[v];
                relax(m[v], d[v], E1, E2, dE1, dE2, v == NV - 1);
            }
        }
    };
    double cp, sp;
    sincos(-(double(a.g_pr) * zz) - dt_pr * dev::TWO_PI * B0, &sp, &cp);

    if (node == MAP_NODES) {  // the state at the first echo (pssfp_kernels.cuh:72-75)
        const double E1i = exp(-dt_inv / T1), E2i = exp(-dt_inv / T2);
        Vec3d m[1] = {{0.0, 0.0, cos(M_PI * B1)}}, d[1][NT];
#pragma unroll
        for (int k = 0; k < NT; k++) d[0][k] = {0.0, 0.0, 0.0};
        if constexpr (TS::b1) d[0][TS::ib1].z = -M_PI * sin(M_PI * B1);
        relax(m[0], d[0], E1i, E2i, dt_inv * k1 * E1i, dt_inv * k2 * E2i, true);
        const double re = a.RF[0].re, im = a.RF[0].im;
        const std::integral_constant<int, 1> one;
        pulse_all(m, d, one, -0.5 * re, -0.5 * im);
        double s, c;
        sincos(-(2.0 * double(a.g_pr) * zz) - dt_pr * dev::TWO_PI * B0, &s, &c);
        precess_all(m[0], d[0], c, s, true);
        pulse_all(m, d, one, re, im);
        precess_all(m[0], d[0], cp, sp, true);
        if (iso < isos) {
            double* o = t.nodes + (1 + NT) * (MAP_NODES * MAP_ENTRIES) * isos + iso;
            o[0] = m[0].x;
            o[isos] = m[0].y;
            o[2 * isos] = m[0].z;
#pragma unroll
            for (int k = 0; k < NT; k++) {
                o[(3 + 3 * k) * isos] = d[0][k].x;
                o[(4 + 3 * k) * isos] = d[0][k].y;
                o[(5 + 3 * k) * isos] = d[0][k].z;
            }
        }
        return;
    }

    Vec3d m[4] = {{1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {0.0, 0.0, 1.0}, {0.0, 0.0, 0.0}}, d[4][NT];
#pragma unroll
    for (int v = 0; v < 4; v++) {
#pragma unroll
        for (int k = 0; k < NT; k++) d[v][k] = {0.0, 0.0, 0.0};
        precess_all(m[v], d[v], cp, sp, v == 3);
    }
    // the pulse phase is taken out (pssfp_map.h): the amplitude is real.  The
    // loop over nodes is the grid's second dimension
    double theta = MAP_SQRT_X[0];
#pragma unroll
    for (int j = 1; j < MAP_NODES; j++) theta = node == j ? MAP_SQRT_X[j] : theta;
    pulse_all(m, d, std::integral_constant<int, 4> {}, train[0] * theta, 0.0);
#pragma unroll
    for (int v = 0; v < 4; v++) precess_all(m[v], d[v], cp, sp, v == 3);
    if (iso >= isos) return;
    const double odd = 1.0 / theta;
    auto store = [&](int map, const Vec3d& x, const Vec3d& y, const Vec3d& z, const Vec3d& c) {
        double* o = t.nodes + (int64_t(map) * MAP_NODES + node) * MAP_ENTRIES * isos + iso;
        o[MXX * isos] = x.x;
        o[MYX * isos] = x.y;
        o[MXY * isos] = y.x;
        o[MYY * isos] = y.y;
        o[MZZ * isos] = z.z;
        o[MCZ * isos] = c.z;
        o[MZX * isos] = x.z * odd;
        o[MZY * isos] = y.z * odd;
        o[MXZ * isos] = z.x * odd;
        o[MYZ * isos] = z.y * odd;
        o[MCX * isos] = c.x * odd;
        o[MCY * isos] = c.y * odd;
    };
    store(0, m[0], m[1], m[2], m[3]);
#pragma unroll
    for (int k = 0; k < NT; k++) store(1 + k, d[0][k], d[1][k], d[2][k], d[3][k]);
}

// grid: nv_block-voxel blocks of the chunk x slice-position groups
template<int MASK, bool PHASED>
__device__ __forceinline__ void pssfp_map_tangents_block(const MapTangentArgs& t, double (*sums)[MAPT_CHUNK][256], double2 (*esums)[MAPT_CHUNK][128]) {
    using TS = TangentSet<MASK>;
    constexpr int NT = TS::nt, NP = TS::planes, LPI = 2 * NT, ISOS = 256 / LPI, PE = 6 / NT;
    const PssfpArgs& a = t.p.a;
    const int tid = threadIdx.x;
    const int block = int(blockIdx.x) % t.p.vblocks, group = int(blockIdx.x) / t.p.vblocks;
    const int v0 = block * t.p.nv_block, nvb = min(t.p.nv_block, t.nv - v0);
    const int z0 = group * t.p.nz_group, nzg = min(t.p.nz_group, a.nz - z0);
    const int64_t isos = int64_t(t.nv) * a.nz;
    // lanes past the block repeat its last isochromat; their sums are not read
    const int local = min(tid / LPI, nvb * nzg - 1);
    const int64_t iso = int64_t(v0 + local / nzg) * a.nz + z0 + local % nzg;
    const int sub = tid % LPI, f = sub >> 1;
    const bool half = sub & 1;

    // Newton coefficients of the lane's six entries of its field's map and of its
    // share of the state's: x's row, or y's, and z's row split between the halves
    constexpr int ROW0[6] = {MXX, MXY, MXZ, MCX, MZX, MZZ}, ROW1[6] = {MYY, MYX, MYZ, MCY, MZY, MCZ};
    double T[6][MAP_NODES], B[PE][MAP_NODES];
#pragma unroll
    for (int e = 0; e < 6; e++) {
        const int entry = half ? ROW1[e] : ROW0[e];
#pragma unroll
        for (int j = 0; j < MAP_NODES; j++)
            T[e][j] = t.nodes[((int64_t(1 + f) * MAP_NODES + j) * MAP_ENTRIES + entry) * isos + iso];
    }
#pragma unroll
    for (int e = 0; e < PE; e++) {
        const int mine = NT == 1 ? e : 3 * f + e;
        int entry = half ? ROW1[0] : ROW0[0];
#pragma unroll
        for (int k = 1; k < 6; k++) entry = mine == k ? (half ? ROW1[k] : ROW0[k]) : entry;
#pragma unroll
        for (int j = 0; j < MAP_NODES; j++) B[e][j] = t.nodes[(int64_t(j) * MAP_ENTRIES + entry) * isos + iso];
    }
#pragma unroll
    for (int o = 1; o < MAP_NODES; o++)
#pragma unroll
        for (int j = MAP_NODES - 1; j >= o; j--) {
            const double inv = 1.0 / (MAP_X[j] - MAP_X[j - o]);
#pragma unroll
            for (int e = 0; e < 6; e++) T[e][j] = (T[e][j] - T[e][j - 1]) * inv;
#pragma unroll
            for (int e = 0; e < PE; e++) B[e][j] = (B[e][j] - B[e][j - 1]) * inv;
        }

    typedef const double __attribute__((address_space(4))) ConstDouble;
    ConstDouble* row = (ConstDouble*)(uintptr_t)(t.p.train + MAP_ROW);
    Vec3d m, d;
    {
        const double* o = t.nodes + (1 + NT) * (MAP_NODES * MAP_ENTRIES) * isos + iso;
        m = {o[0], o[isos], o[2 * isos]};
        d = {o[(3 + 3 * f) * isos], o[(4 + 3 * f) * isos], o[(5 + 3 * f) * isos]};
        if constexpr (PHASED) {  // into the frame of TR 0's pulse
            rotate_z(m, row[MAP_PHASE + 2], row[MAP_PHASE + 3]);
            rotate_z(d, row[MAP_PHASE + 2], row[MAP_PHASE + 3]);
        }
    }
    // own and other transverse component, and z, of the state and of the tangent
    double mo = half ? m.y : m.x, mt = half ? m.x : m.y, mz = m.z;
    double dox = half ? d.y : d.x, dt = half ? d.x : d.y, dz = d.z;
    const double turn = half ? 1.0 : -1.0;  // sign of the other component in a turn about z
    double next[MAP_NODES];
#pragma unroll
    for (int j = 0; j < MAP_NODES; j++) next[j] = row[j];

    int per = 1;
    while (per < 32 && per * 2 * nvb * NP <= 32) per *= 2;
    const size_t nv_all = size_t(a.tissue.nvoxels), plane = size_t(a.nTR) * nv_all;
    auto write_sums = [&](int n0, int count, int buf) {
        // in a pass of one field formed anew for each chunk: kept, they take the
        // registers that make it spill (pssfp_map.hip says why no kernel may)
        int lane = tid;
        if constexpr (NT == 1) asm volatile("" : "+v"(lane));
        const int sum_tr = lane >> 5, sum_t = lane & 31;
        const int n = n0 + sum_tr;
        for (int w = sum_t / per; w < nvb * NP; w += 32 / per) {
            const int vox = w / NP, k = w % NP;  // plane k: the echoes, then the fields
            const bool echo = TS::echo && k == 0;
            const int field = k - int(TS::echo);
            double x = 0.0, y = 0.0;
            if (sum_tr < count) {
                for (int i = sum_t % per; i < nzg; i += per) {
                    const int at = vox * nzg + i;
                    const double2 e = echo ? esums[buf][sum_tr][at]
                                           : *reinterpret_cast<const double2*>(&sums[buf][sum_tr][at * LPI + 2 * max(field, 0)]);
                    x += e.x;
                    y += e.y;
                }
            }
            for (int off = 1; off < per; off <<= 1) {
                x += __shfl_xor(x, off);
                y += __shfl_xor(y, off);
            }
            if (sum_tr < count && sum_t % per == 0) {
                if constexpr (PHASED) {  // back from the pulse's frame
                    const double* r = t.p.train + size_t(n + 1) * MAP_ROW + MAP_PHASE + 2;
                    const double xr = r[0] * x + r[1] * y;
                    y = r[0] * y - r[1] * x;
                    x = xr;
                }
                const size_t at = size_t(n) * nv_all + t.v0 + v0 + vox;
                if (t.p.groups == 1) {
                    cfloat* o = k == 0 ? t.out[0] : k == 1 ? t.out[1] : t.out[2];
                    o[at] = {float(x), float(y)};
                } else {
                    reinterpret_cast<double2*>(t.p.partial)[(size_t(group) * NP + k) * plane + at] = make_double2(x, y);
                }
            }
        }
    };

    int buf = 0;
    for (int n0 = 0; n0 < a.nTR; n0 += MAPT_CHUNK) {
        const int count = min(MAPT_CHUNK, a.nTR - n0);
        for (int i = 0; i < count; i++) {
            double x[MAP_NODES];
#pragma unroll
            for (int j = 0; j < MAP_NODES; j++) x[j] = next[j];
            if constexpr (PHASED) {
                if (n0 + i > 0) {
                    const double c = row[MAP_PHASE], s = turn * row[MAP_PHASE + 1];
                    const double o = fma(c, mo, s * mt), p = fma(c, dox, s * dt);
                    mt = fma(c, mt, -s * mo);
                    dt = fma(c, dt, -s * dox);
                    mo = o;
                    dox = p;
                }
            }
            row += MAP_ROW;
#pragma unroll
            for (int j = 0; j < MAP_NODES; j++) next[j] = row[j];
            if (n0 + i > 0) {
                const double theta = x[0];
                double e[6], g[6], s[PE];
#pragma unroll
                for (int q = 0; q < PE; q++) s[q] = B[q][MAP_NODES - 1];
#pragma unroll
                for (int q = 0; q < 6; q++) g[q] = T[q][MAP_NODES - 1];
#pragma unroll
                for (int j = MAP_NODES - 2; j >= 0; j--) {
#pragma unroll
                    for (int q = 0; q < PE; q++) s[q] = fma(s[q], x[1 + j], B[q][j]);
#pragma unroll
                    for (int q = 0; q < 6; q++) g[q] = fma(g[q], x[1 + j], T[q][j]);
                }
                if constexpr (NT == 1) {
#pragma unroll
                    for (int q = 0; q < 6; q++) e[q] = s[q];
                } else {  // from the lane of field 0, and of field 1, of the same half
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        e[q] = quad<0x44>(s[q]);
                        e[3 + q] = quad<0xEE>(s[q]);
                    }
                }
                const double h = half ? 1.0 : mz, dh = half ? 0.0 : dz;
                const double no = fma(theta, fma(e[2], mz, e[3]), fma(e[0], mo, e[1] * mt));
                const double nz = fma(theta, e[4] * mo, e[5] * h);
                const double po = fma(theta, fma(e[2], dz, fma(g[2], mz, g[3])),
                                      fma(e[0], dox, fma(e[1], dt, fma(g[0], mo, g[1] * mt))));
                const double pz = fma(theta, fma(e[4], dox, g[4] * mo), fma(e[5], dh, g[5] * h));
                mo = no;
                mt = quad<0xB1>(no);
                mz = nz + quad<0xB1>(nz);
                dox = po;
                dt = quad<0xB1>(po);
                dz = pz + quad<0xB1>(pz);
            }
            sums[buf][i][tid] = dox;
            if constexpr (TS::echo) {
                if (f == 0) reinterpret_cast<double*>(&esums[buf][i][tid / LPI])[half] = mo;
            }
        }
        __syncthreads();
        write_sums(n0, count, buf);
        buf ^= 1;
    }
}

template<int MASK>
__global__ void __launch_bounds__(256, 2) pssfp_map_tangents(MapTangentArgs t) {
    constexpr bool ECHO = TangentSet<MASK>::echo;
    __shared__ __align__(16) double sums[2][MAPT_CHUNK][256];
    __shared__ double2 esums[ECHO ? 2 : 1][ECHO ? MAPT_CHUNK : 1][128];
    if (t.p.train[1] == 0.0) return;  // pssfp_iso_tangents runs instead
    double2(*e)[MAPT_CHUNK][128] = reinterpret_cast<double2(*)[MAPT_CHUNK][128]>(&esums[0][0][0]);
    if (t.p.train[2] != 0.0) {
        pssfp_map_tangents_block<MASK, true>(t, sums, e);
    } else {
        pssfp_map_tangents_block<MASK, false>(t, sums, e);
    }
}

}  // namespace kernels

namespace {

using namespace kernels;

template<int MASK>
void run_pass(const CompasContext& ctx, const PssfpArgs& a, const double* train, cfloat* const* planes) {
    constexpr int NT = TangentSet<MASK>::nt, NP = TangentSet<MASK>::planes;
    MapTangentArgs t {};
    t.p.a = a;
    t.p.train = train;
    for (int k = 0; k < NP; k++) t.out[k] = planes[k];
    // a further group has to raise the isochromats in use by a twenty-fifth
    const PssfpWorkgroup w = pssfp_workgroup(a.nz, 128 / NT, 128 / NT, 0.04);
    COMPAS_CHECK(w.groups > 0);
    t.p.nv_block = w.nv_block;
    t.p.nz_group = w.nz_group;
    t.p.groups = w.groups;
    const int64_t plane = int64_t(a.nTR) * a.tissue.nvoxels;
    Array<cfloat, 2> part;
    if (t.p.groups > 1) part = ctx.empty<cfloat, 2>({int64_t(pssfp_map_partial_planes(t.p)) * NP, plane});
    t.p.partial = part.data();
    // node values of at most about 1 GiB of isochromats at a time
    const int64_t per_iso = int64_t((1 + NT) * MAP_NODES * MAP_ENTRIES + 3 + 3 * NT) * 8;
    const int chunk = int(std::min<int64_t>(a.tissue.nvoxels, std::max<int64_t>(1, (int64_t(1) << 30) / (per_iso * a.nz))));
    auto nodes = ctx.empty<double, 1>({per_iso / 8 * chunk * a.nz});
    t.nodes = nodes.data();
    for (int v0 = 0; v0 < a.tissue.nvoxels; v0 += chunk) {
        t.v0 = v0;
        t.nv = std::min(chunk, a.tissue.nvoxels - v0);
        t.p.vblocks = int(dev::div_ceil(t.nv, t.p.nv_block));
        {
            KernelScope ks(ctx, "pssfp_map_nodes");
            pssfp_map_nodes<MASK><<<dim3(dev::div_ceil(int64_t(t.nv) * a.nz, int64_t(256)), MAP_NODES + 1), 256, 0, ctx.stream()>>>(t);
            check_launch("pssfp_map_nodes");
        }
        KernelScope ks(ctx, "pssfp_map_tangents");
        pssfp_map_tangents<MASK><<<unsigned(t.p.vblocks * t.p.groups), 256, 0, ctx.stream()>>>(t);
        check_launch("pssfp_map_tangents");
    }
    for (int k = 0; k < NP; k++)
        pssfp_map_sum(ctx, planes[k], part.data() + 2 * k * plane, t.p.groups, plane, NP * plane, train);
}

}  // namespace

// FP64 operations per isochromat: direct, RF sub-step and TR; maps, TR and (a
// node's) RF sub-step.  At 8 sub-steps and 64 to 100 TRs all four fields take
// the same time either way (0.96 and 1.41 ms at 5000 voxels x 35 positions, by
// sub-steps); T1 + T2 at 12 and 64 0.60 and 0.55 ms.
bool pssfp_map_tangents_pay(int mask, int nTR, int nRF) {
    if (nRF < 1 || nRF > RF_CHUNK) return false;
    double direct, per_tr, per_step;
    switch (mask & ~TM_ECHO) {
        case TM_T1 | TM_T2 | TM_B1 | TM_B0: direct = 155, per_tr = 912, per_step = 520; break;
        case TM_T1 | TM_T2: direct = 88, per_tr = 456, per_step = 180; break;
        case TM_B1:
        case TM_B0: direct = 110, per_tr = 250, per_step = 220; break;
        default: direct = 65, per_tr = 250, per_step = 130; break;
    }
    return nTR * per_tr + MAP_NODES * per_step * nRF + 5000.0 < 0.9 * direct * double(nTR) * nRF;
}

void launch_pssfp_map_tangents(const CompasContext& ctx, int mask, const PssfpArgs& a, const double* train, cfloat* const* planes) {
    const int echo = mask & TM_ECHO ? 1 : 0;
    switch (mask) {
        case TM_T1: run_pass<TM_T1>(ctx, a, train, planes); break;
        case TM_T2: run_pass<TM_T2>(ctx, a, train, planes); break;
        case TM_B1: run_pass<TM_B1>(ctx, a, train, planes); break;
        case TM_B0: run_pass<TM_B0>(ctx, a, train, planes); break;
        case TM_T1 | TM_T2: run_pass<TM_T1 | TM_T2>(ctx, a, train, planes); break;
        case TM_T1 | TM_T2 | TM_ECHO: run_pass<TM_T1 | TM_T2 | TM_ECHO>(ctx, a, train, planes); break;
        case TM_T1 | TM_T2 | TM_B1 | TM_B0:
        case TM_T1 | TM_T2 | TM_B1 | TM_B0 | TM_ECHO:
            if (echo) run_pass<TM_T1 | TM_T2 | TM_ECHO>(ctx, a, train, planes);
            else run_pass<TM_T1 | TM_T2>(ctx, a, train, planes);
            run_pass<TM_B1 | TM_B0>(ctx, a, train, planes + 2 + echo);
            break;
        default: COMPAS_ERROR("no tangent kernel for this field set");
    }
}

}  // namespace compas
