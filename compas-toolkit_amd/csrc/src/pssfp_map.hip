// pSSFP simulation with one affine map per isochromat and TR (gfx950).
//
// Stepping through the nRF RF sub-steps costs about 31 nRF FP64 operations
// per isochromat and TR; the map of a whole TR is a function of the flip angle
// alone (pssfp_map.h), so this kernel finds its twelve entries once per
// isochromat at MAP_NODES flip angles and in every TR evaluates twelve
// polynomials of degree MAP_NODES - 1 in Newton's form, 84 FMAs, plus 12 to
// apply them.
//
// Design (MI355X):
//   * One isochromat per lane: its 96 Newton coefficients take 192 VGPRs and
//     stay there for the whole train, two waves per SIMD, without a spill (50176
//     voxels x 1120 TRs x 35 positions 8.8 ms; 9.3 with 193 spills in the set-up).  The twelve Horner
//     chains are independent, which hides the FMA latency.  Their common
//     factors x_n - x_j are the same for every isochromat: wave-uniform, so
//     scalar loads from the train's table feed SGPR operands.
//   * A workgroup of 256 lanes holds nv_block voxels x nz_group slice
//     positions, so the sum over slice positions stays in it: each lane puts
//     its transverse magnetisation into LDS, and every MAP_CHUNK TRs the
//     workgroup adds up the previous chunk (FP64, in order of position) while
//     it computes the next; two LDS buffers, one barrier per chunk.  No partial
//     echoes go through HBM unless there are more than about eighty slice
//     positions; then each group has an FP64 plane.
//   * Neighbouring voxel blocks run on one XCD, so that the 8 nv_block bytes a
//     workgroup writes per TR meet their neighbours' in that XCD's L2.
//   * What bounds it: FP64 issue.  At 50176 voxels x 1120 TRs x 35 positions the
//     VALU is busy 79% of the cycles (148 k instructions per wave, 13% of them
//     the set-up); the rest is the waits around the chunk sums.
//   * Whether a train is within MAP_MAX_TYPE is found on the device: the train
//     lives there and may be rewritten between calls.  The sub-step kernel is
//     launched after this one, and one of the two leaves at once (the request
//     server reads the answer back and cuts the sub-steps into work items).

#include <algorithm>

#include "compas/device/common.h"
#include "compas/device/pssfp_common.h"
#include "compas/device/pssfp_map.h"
#include "compas/internal.h"
#include "compas/pssfp_layout.h"

namespace compas {
namespace kernels {

constexpr int MAP_CHUNK = 8;  // TRs summed over slice positions at a time

// The train's table (pssfp_map.h).  One workgroup of 1024 threads.
__global__ void __launch_bounds__(1024) pssfp_map_train(PssfpArgs a, double* train) {
    __shared__ double s_rf[1024], s_b1[1024], s_g[1024];
    __shared__ int s_phase;
    const int tid = threadIdx.x;
    if (tid == 0) s_phase = 0;
    // a NaN must not be dropped by a maximum: it is counted as infinite
    auto larger = [](double m, double v) { return v <= m ? m : (v == v ? v : HUGE_VAL); };
    double rf = 0.0, b1 = 0.0, g = 0.0;
    bool phase = false;
    for (int n = tid; n < a.nTR; n += 1024) {
        rf = larger(rf, hypot(double(a.RF[n].re), double(a.RF[n].im)));
        phase = phase || a.RF[n].im != 0.0f;
    }
#pragma unroll 8
    for (int v = tid; v < a.tissue.nvoxels; v += 1024) b1 = larger(b1, fabs(double(a.tissue.B1(v))));
    for (int k = tid; k < a.nRF; k += 1024) g += hypot(double(a.gamma_dt_RF[k].re), double(a.gamma_dt_RF[k].im));
    s_rf[tid] = rf;
    s_b1[tid] = b1;
    s_g[tid] = g;
    __syncthreads();
    if (phase) s_phase = 1;
    for (int off = 512; off > 0; off >>= 1) {
        if (tid < off) {
            s_rf[tid] = larger(s_rf[tid], s_rf[tid + off]);
            s_b1[tid] = larger(s_b1[tid], s_b1[tid + off]);
            s_g[tid] += s_g[tid + off];
        }
        __syncthreads();
    }
    const double top = s_rf[0];
    const double unit = top > 0.0 ? 1.0 / top : 0.0;
    const bool phased = s_phase != 0;
    if (tid == 0) {
        train[0] = top;
        train[1] = top * s_g[0] * s_b1[0] <= MAP_MAX_TYPE ? 1.0 : 0.0;
        train[2] = phased ? 1.0 : 0.0;
    }
    // amplitude and unit phase; a real train keeps its signs in the amplitude
    auto entry = [&](int n, double& theta, double& c, double& s) {
        const double re = a.RF[n].re, im = a.RF[n].im;
        theta = re;
        c = 1.0;
        s = 0.0;
        if (phased) {
            theta = hypot(re, im);
            if (theta > 0.0) {
                c = re / theta;
                s = im / theta;
            }
        }
        theta *= unit;
    };
    for (int n = tid; n < a.nTR; n += 1024) {
        double* row = train + size_t(n + 1) * MAP_ROW;
        double theta, c, s, t0, c0 = 1.0, s0 = 0.0;
        entry(n, theta, c, s);
        if (n > 0) entry(n - 1, t0, c0, s0);
        row[0] = theta;
#pragma unroll
        for (int j = 0; j < MAP_NODES - 1; j++) row[1 + j] = fma(theta, theta, -MAP_X[j]);
        row[MAP_PHASE] = c * c0 + s * s0;
        row[MAP_PHASE + 1] = s * c0 - c * s0;
        row[MAP_PHASE + 2] = c;
        row[MAP_PHASE + 3] = s;
    }
}

// One RF pulse of amplitude rf: nv vectors through the sub-steps, the last of
// them with regrowth (the others are the columns of the linear part)
template<int NV>
__device__ __forceinline__ void pulse(const IsoConst& k, const double2* grf, int nRF, double re, double im, Vec3d (&m)[NV]) {
    const SeriesConst series;
    for (int i = 0; i < nRF; i++) {
        const double2 g = grf[i];
        const double ax = (re * g.x - im * g.y) * k.B1, ay = -(re * g.y + im * g.x) * k.B1;
        double M[9];
        substep_matrix(series, ax, ay, k.az, k.E1, k.E2, M);
#pragma unroll
        for (int v = 0; v < NV; v++) apply3(M, m[v]);
        m[NV - 1].z += k.R1;
    }
}

// The echoes of nv_block voxels x nz_group slice positions; `block` and `group`
// name them.
template<bool PHASED>
__device__ __forceinline__ void pssfp_map_block(
    const PssfpMapArgs& p, int block, int group, const double2* grf, double2 (*sums)[MAP_CHUNK][256]) {
    const PssfpArgs& a = p.a;
    const int tid = threadIdx.x;
    const int nv = a.tissue.nvoxels;
    const int v0 = block * p.nv_block, nvb = min(p.nv_block, nv - v0);
    const int z0 = group * p.nz_group, nzg = min(p.nz_group, a.nz - z0);
    // lanes past the block repeat its last isochromat; their sums are not read
    const int iso = min(tid, nvb * nzg - 1);
    const int voxel = v0 + iso / nzg;
    const double zz = a.z[z0 + iso % nzg];

    IsoConst k;
    const double T1 = a.tissue.T1(voxel), T2 = a.tissue.T2(voxel), B0 = a.tissue.B0(voxel);
    k.B1 = a.tissue.B1(voxel);
    k.E1 = exp(-double(a.dt_ex) / T1);
    k.E2 = exp(-double(a.dt_ex) / T2);
    k.R1 = 1.0 - k.E1;
    k.az = -(double(a.g_ex) * zz) - double(a.dt_ex) * dev::TWO_PI * B0;
    const double off_pr = double(a.dt_pr) * dev::TWO_PI * B0;
    const double E2_pr = exp(-double(a.dt_pr) / T2);
    k.P1 = exp(-double(a.dt_pr) / T1);
    k.Q1 = 1.0 - k.P1;
    sincos(-(double(a.g_pr) * zz) - off_pr, &k.ps, &k.pc);
    k.ps *= E2_pr;
    k.pc *= E2_pr;

    // inversion, the alpha/2 pulse with the doubled prephaser, and the first TR
    // by their sub-steps (pssfp_kernels.cuh:72-75)
    Vec3d s[1] = {{0.0, 0.0, 0.0}};
    {
        const double E1_inv = exp(-double(a.dt_inv) / T1);
        s[0].z = fma(cos(M_PI * k.B1), E1_inv, 1.0 - E1_inv);
        const double re = a.RF[0].re, im = a.RF[0].im;
        pulse(k, grf, a.nRF, -0.5 * re, -0.5 * im, s);
        double ss, cc;
        sincos(-(2.0 * double(a.g_pr) * zz) - off_pr, &ss, &cc);
        rotate_z(s[0], cc, ss);
        relax3(s[0], k.P1, E2_pr, k.Q1);
        pulse(k, grf, a.nRF, re, im, s);
        precess(k, s[0], k.Q1);
    }
    // Newton coefficients of the twelve entries.  Those of the first nodes wait in
    // the lane's slots of the sums until the last node has been through its pulse:
    // with all in registers the pulse spills, and a kernel with scratch memory is
    // aborted where the device's memory is taken when it is launched
    const double* train = p.train;
    const double top = train[0];
    constexpr int WAIT = 2;  // nodes, six slots each of 2 MAP_CHUNK
    double C[MAP_ENTRIES][MAP_NODES];
#pragma unroll
    for (int j = 0; j < MAP_NODES; j++) {
        Vec3d m[4] = {{k.pc, k.ps, 0.0}, {-k.ps, k.pc, 0.0}, {0.0, 0.0, k.P1}, {0.0, 0.0, k.Q1}};
        pulse(k, grf, a.nRF, top * MAP_SQRT_X[j], 0.0, m);
#pragma unroll
        for (int v = 0; v < 4; v++) precess(k, m[v], v == 3 ? k.Q1 : 0.0);
        const double odd = 1.0 / MAP_SQRT_X[j];
        C[MXX][j] = m[0].x;
        C[MYX][j] = m[0].y;
        C[MXY][j] = m[1].x;
        C[MYY][j] = m[1].y;
        C[MZZ][j] = m[2].z;
        C[MCZ][j] = m[3].z;
        C[MZX][j] = m[0].z * odd;
        C[MZY][j] = m[1].z * odd;
        C[MXZ][j] = m[2].x * odd;
        C[MYZ][j] = m[2].y * odd;
        C[MCX][j] = m[3].x * odd;
        C[MCY][j] = m[3].y * odd;
        if (j < WAIT) {
#pragma unroll
            for (int q = 0; q < 6; q++) {
                const int slot = 6 * j + q;
                sums[slot / MAP_CHUNK][slot % MAP_CHUNK][tid] = make_double2(C[2 * q][j], C[2 * q + 1][j]);
            }
            asm volatile("" ::: "memory");  // the values live there from here on
        }
    }
#pragma unroll
    for (int j = 0; j < WAIT; j++)
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const int slot = 6 * j + q;
            const double2 v = sums[slot / MAP_CHUNK][slot % MAP_CHUNK][tid];
            C[2 * q][j] = v.x;
            C[2 * q + 1][j] = v.y;
        }
    // divided differences, one entry after the other: all at once they spill
#pragma unroll
    for (int e = 0; e < MAP_ENTRIES; e++) {
#pragma unroll
        for (int o = 1; o < MAP_NODES; o++)
#pragma unroll
            for (int j = MAP_NODES - 1; j >= o; j--) C[e][j] = (C[e][j] - C[e][j - 1]) * (1.0 / (MAP_X[j] - MAP_X[j - o]));
        __builtin_amdgcn_sched_barrier(0);
    }

    Vec3d m = s[0];
    // the table's rows are read through the constant address space: the same
    // address in every lane, so scalar loads, each a TR before its use
    typedef const double __attribute__((address_space(4))) ConstDouble;
    ConstDouble* row = (ConstDouble*)(uintptr_t)(train + MAP_ROW);
    if constexpr (PHASED) rotate_z(m, row[MAP_PHASE + 2], row[MAP_PHASE + 3]);  // into the frame of TR 0's pulse
    double next[MAP_NODES];
#pragma unroll
    for (int j = 0; j < MAP_NODES; j++) next[j] = row[j];

    // threads of one TR's sum: MAP_CHUNK x 32; several per voxel where there are
    // few (reading ahead, or spreading the reads over the next chunk's TRs,
    // took more instructions than the wait it saved)
    const int sum_tr = tid >> 5, sum_t = tid & 31;
    int per = 1;
    while (per < 32 && per * 2 * nvb <= 32) per *= 2;
    auto write_sums = [&](int n0, int count, int buf) {
        const int n = n0 + sum_tr;
        for (int w = sum_t / per; w < nvb; w += 32 / per) {
            double x = 0.0, y = 0.0;
            if (sum_tr < count) {
                for (int i = sum_t % per; i < nzg; i += per) {
                    const double2 e = sums[buf][sum_tr][w * nzg + i];
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
                    const double* r = train + size_t(n + 1) * MAP_ROW + MAP_PHASE + 2;
                    const double xr = r[0] * x + r[1] * y;
                    y = r[0] * y - r[1] * x;
                    x = xr;
                }
                const size_t at = size_t(n) * nv + v0 + w;
                if (p.groups == 1) {
                    a.echos[at] = {float(x), float(y)};
                } else {
                    reinterpret_cast<double2*>(p.partial)[size_t(group) * a.nTR * nv + at] = make_double2(x, y);
                }
            }
        }
    };

    int buf = 0;
    for (int n0 = 0; n0 < a.nTR; n0 += MAP_CHUNK) {
        const int count = min(MAP_CHUNK, a.nTR - n0);
        for (int i = 0; i < count; i++) {
            double d[MAP_NODES];
#pragma unroll
            for (int j = 0; j < MAP_NODES; j++) d[j] = next[j];
            if (n0 + i > 0) {
                if constexpr (PHASED) rotate_z(m, row[MAP_PHASE], row[MAP_PHASE + 1]);
            }
            row += MAP_ROW;
#pragma unroll
            for (int j = 0; j < MAP_NODES; j++) next[j] = row[j];
            if (n0 + i > 0) {
                const double theta = d[0];
                double e[MAP_ENTRIES];
#pragma unroll
                for (int q = 0; q < MAP_ENTRIES; q++) e[q] = C[q][MAP_NODES - 1];
#pragma unroll
                for (int j = MAP_NODES - 2; j >= 0; j--) {
#pragma unroll
                    for (int q = 0; q < MAP_ENTRIES; q++) e[q] = fma(e[q], d[1 + j], C[q][j]);
                }
                const double x = fma(e[MXX], m.x, fma(e[MXY], m.y, theta * fma(e[MXZ], m.z, e[MCX])));
                const double y = fma(e[MYX], m.x, fma(e[MYY], m.y, theta * fma(e[MYZ], m.z, e[MCY])));
                const double z = fma(e[MZZ], m.z, fma(theta, fma(e[MZX], m.x, e[MZY] * m.y), e[MCZ]));
                m = {x, y, z};
            }
            sums[buf][i][tid] = make_double2(m.x, m.y);
        }
        __syncthreads();
        write_sums(n0, count, buf);
        buf ^= 1;
    }
}

// Workgroup b of the launch, or item (job, unit) = items[b] of a work table:
// unit u is voxel block u % vblocks of slice-position group u / vblocks.
__global__ void __launch_bounds__(256, 2) pssfp_map(
    PssfpMapArgs single, const PssfpMapArgs* __restrict__ jobs, const int2* __restrict__ items) {
    __shared__ double2 grf[RF_CHUNK];
    __shared__ double2 sums[2][MAP_CHUNK][256];
    PssfpMapArgs p = single;
    int unit = int(blockIdx.x);
    if (items != nullptr) {
        p = jobs[items[blockIdx.x].x];
        unit = items[blockIdx.x].y;
    } else {
        // consecutive workgroups go to the XCDs in turn: give each XCD a run of
        // neighbouring units
        const int per = int(gridDim.x) / 8;
        if (unit < 8 * per) unit = (unit % 8) * per + unit / 8;
    }
    if (p.train[1] == 0.0) return;  // pssfp_iso runs instead
    for (int i = threadIdx.x; i < p.a.nRF; i += 256) grf[i] = make_double2(double(p.a.gamma_dt_RF[i].re), double(p.a.gamma_dt_RF[i].im));
    __syncthreads();
    const int group = unit / p.vblocks;
    if (p.train[2] != 0.0) {
        pssfp_map_block<true>(p, unit % p.vblocks, group, grf, sums);
    } else {
        pssfp_map_block<false>(p, unit % p.vblocks, group, grf, sums);
    }
}

// out[i] = sum over the groups' planes (plane j at partial + j stride), in
// order; nothing where the maps did not serve the train
__global__ void pssfp_map_sum(
    cfloat* __restrict__ out, const double2* __restrict__ partial, int groups, int64_t n, int64_t stride,
    const double* train) {
    if (train[1] == 0.0) return;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
        double re = 0.0, im = 0.0;
        for (int j = 0; j < groups; j++) {
            const double2 q = partial[size_t(j) * size_t(stride) + size_t(i)];
            re += q.x;
            im += q.y;
        }
        out[i] = {float(re), float(im)};
    }
}

}  // namespace kernels

// Whether the maps pay for a train: per isochromat the sub-steps cost about
// 31 nRF + 16 FP64 operations in every TR, the maps 100 and their set-up 80
// nRF at each node.  Measured at 50176 voxels x 35 positions x 25 sub-steps:
// sub-steps 50 us per TR, maps 6.5 us per TR after 1.3 ms of set-up, so 64 TRs
// take 3.2 ms by sub-steps and 1.7 ms by maps; 1120 TRs 54.8 and 9.3 ms.
bool pssfp_map_pays(int nTR, int nRF) {
    if (nRF < 1 || nRF > kernels::RF_CHUNK) return false;
    const double direct = double(nTR) * (31.0 * nRF + 16.0);
    const double maps = double(nTR) * 100.0 + kernels::MAP_NODES * 80.0 * nRF + 62.0 * nRF + 1500.0;
    return maps < 0.9 * direct;
}

int64_t pssfp_map_train_size(int nTR) {
    return int64_t(nTR + 2) * kernels::MAP_ROW;  // the header, the rows, and one read ahead
}

void pssfp_map_table(const CompasContext& ctx, const kernels::PssfpArgs& a, double* train) {
    KernelScope ks(ctx, "pssfp_map_train");
    kernels::pssfp_map_train<<<1, 1024, 0, ctx.stream()>>>(a, train);
    check_launch("pssfp_map_train");
}

void pssfp_map_setup(const CompasContext& ctx, kernels::PssfpMapArgs& p, const kernels::PssfpArgs& a, double* train, int zpl) {
    p.a = a;
    p.train = train;
    p.partial = nullptr;
    // at least two voxels to a workgroup; a further group has to raise the lanes
    // in use by a tenth
    const PssfpWorkgroup w = pssfp_workgroup(a.nz, 256, 128, 0.1);
    COMPAS_CHECK(w.groups > 0);
    p.nv_block = w.nv_block;
    p.nz_group = w.nz_group;
    p.groups = w.groups;
    p.vblocks = int(dev::div_ceil(a.tissue.nvoxels, p.nv_block));
    p.direct_zpl = zpl;
    p.direct_groups = (a.nz + zpl - 1) / zpl;
    pssfp_map_table(ctx, a, train);
}

int pssfp_map_partial_planes(const kernels::PssfpMapArgs& p) {
    return p.groups > 1 ? 2 * p.groups : 0;
}

int64_t pssfp_map_units(const kernels::PssfpMapArgs& p) {
    return int64_t(p.vblocks) * p.groups;
}

void launch_pssfp_map(
    const CompasContext& ctx, const kernels::PssfpMapArgs& single, const kernels::PssfpMapArgs* jobs,
    const int2* items, int64_t n) {
    if (n <= 0) return;
    KernelScope ks(ctx, jobs ? "pssfp_map_table" : "pssfp_map");
    kernels::pssfp_map<<<unsigned(n), 256, 0, ctx.stream()>>>(single, jobs, items);
    check_launch("pssfp_map");
}

void pssfp_map_sum(
    const CompasContext& ctx, cfloat* out, const cfloat* partial, int groups, int64_t n, int64_t stride,
    const double* train) {
    if (groups <= 1 || n == 0) return;
    KernelScope ks(ctx, "pssfp_map_sum");
    const int64_t blocks = std::min<int64_t>(dev::div_ceil(n, int64_t(256)), 8192);
    kernels::pssfp_map_sum<<<unsigned(blocks), 256, 0, ctx.stream()>>>(
        out, reinterpret_cast<const double2*>(partial), groups, n, stride, train);
    check_launch("pssfp_map_sum");
}

void pssfp_map_finish(const CompasContext& ctx, const kernels::PssfpMapArgs& p) {
    const int64_t n = int64_t(p.a.nTR) * p.a.tissue.nvoxels;
    pssfp_map_sum(ctx, p.a.echos, p.partial, p.groups, n, n, p.train);
    launch_pssfp_unmapped(ctx, p);
    pssfp_sum_groups(ctx, p.a.echos, p.partial, p.direct_groups - 1, n, n, p.train);
}

}  // namespace compas
