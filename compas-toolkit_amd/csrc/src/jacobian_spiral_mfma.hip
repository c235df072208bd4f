// J^H.y on the spiral trajectory (six parameters) with the sample sums on MFMA.
//
// Per readout r the adjoint needs, for every voxel v and coil c,
//   U[c][v]  = sum_s y[c][r][s] conj(Phi[r][s][v])
//   U'[c][v] = sum_s (s - ns/2) y[c][r][s] conj(Phi[r][s][v])
// (jacobian_spiral.hip states Phi and how U, U' combine into the six rows).
// Phi is a geometric sequence in s: with s = sb + S t + n, n < S = 8 KS, Phi_s =
// Phi_sb E^(S t) E^n and
//   U  = conj(Phi_sb) sum_t conj(E^(S t)) G_t,   G_t  = sum_n y_s conj(E^n)
//   U' = conj(Phi_sb) sum_t conj(E^(S t)) G'_t,  G'_t = sum_n (s - ns/2) y_s conj(E^n).
// (s - ns/2 in one piece: split as (sb + S t - ns/2) G_t + sum_n n y_s conj(E^n) its
// two terms cancel near the centre of the readout, where a readout peaks, after
// each has been rounded.)  G and G' are a complex GEMM, rows (coil, t) x K = n x N = voxels, whose B
// operand has S generated elements per voxel and readout instead of ns; the
// sums over t are Horner's rule on the accumulators.  It runs on
// v_mfma_f32_32x32x16_bf16 with BF16 hi + lo operands (FP32 accumulation):
//   * A: four row tiles (real and imaginary parts of G and of G') of 32 (coil,
//     t) rows, written once per call in fragment order by spiral_y_fragments
//     and copied to LDS per readout, the next readout's behind the current one;
//   * B: lane l holds voxel l % 32 and samples n = 8 ks + 4 (l / 32) + j of K
//     step ks, advanced by E^8 per step, in registers; T tiles of 32 voxels per
//     wave share the A fragments;
//   * the rows are ordered so that a lane's sixteen accumulator elements are
//     two coils with T8's eight t each, or four coils with four: the sums over
//     t and over the lane's coils (with conj(C)) need no exchange, and the
//     products with conj(m) and conj(dm_p) are done once per readout.
// Sample blocks of S T and coil groups repeat the two stages within a readout.
//
// What bounds it: MFMA (47% of the cycles) and VALU (51%) issue, which overlap
// little because a barrier per readout keeps the waves of a CU in step, at 2.0
// GHz.  50176 voxels x 1120 readouts x 512 samples, 4 coils: 14.9 -> 5.5 ms
// against a form that generated every sample's element; 20000 x 500 x 128 854
// -> 670 us, x 16 452 -> 351 us.
//
// Layout of v_mfma_f32_32x32x16_bf16 (wave64): lane l supplies row (A) or
// column (B) l % 32 and K elements 8 (l / 32) .. + 7; result element e of lane l
// is row 8 (e / 4) + 4 (l / 32) + e % 4, column l % 32.

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "compas/device/common.h"
#include "compas/device/mfma_tile.h"
#include "compas/device/spiral_phasor.h"
#include "compas/internal.h"
#include "compas/spiral_layout.h"

namespace compas {
namespace kernels {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int SHM_TILES = 4;  // row tiles: G_re, G_im, G'_re, G'_im

// Coil (of its group) and t of row tile row `row`
template<bool T8>
__device__ __forceinline__ void shm_row(int row, int& c, int& t) {
    const int a = row >> 3, h = (row >> 2) & 1, b = row & 3;
    c = T8 ? 2 * h + (a >> 1) : 4 * h + a;
    t = T8 ? 4 * (a & 1) + b : b;
}

// A fragments frag[readout][block][K step][tile][hi, lo][lane], block = sample
// block x coil group; grid (nr + ceil(nv / (64 KS)), blocks), block 64 KS.  The
// workgroups after the first nr of a row write the voxels' constants.
template<int KS, bool T8, bool LO>
__global__ void __launch_bounds__(64 * KS) spiral_y_fragments(
    const cfloat* __restrict__ y, int nc, int nr, int ns, int groups, uint4* __restrict__ frag,
    dev::TissueView tissue, float dt, SpiralVoxel* __restrict__ voxels) {
    constexpr int P = LO ? mfma::P_BF16X3 : mfma::P_BF16X1;
    constexpr int S = 8 * KS, T = T8 ? 8 : 4, COILS = T8 ? 4 : 8, PARTS = LO ? 2 : 1;
    const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
    const int r = blockIdx.x, block = blockIdx.y;
    if (r >= nr) {
        const int v = (r - nr) * (64 * KS) + int(threadIdx.x);
        if (block == 0 && v < tissue.nvoxels) voxels[v] = spiral_voxel(tissue, dt, v);
        return;
    }
    int c, t;
    shm_row<T8>(lane & 31, c, t);
    c += COILS * (block % groups);
    const int n0 = 8 * ks + 4 * (lane >> 5);
    const int s0 = (block / groups) * (S * T) + S * t + n0;
    uint32_t hi[SHM_TILES][4], lo[SHM_TILES][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        cfloat v = {0.0f, 0.0f};
        if (c < nc && s0 + j < ns) v = y[(size_t(c) * nr + r) * ns + s0 + j];
        const cfloat w = v * (float(s0 + j) - 0.5f * float(ns));
        mfma::split_pair<P>(v.re, v.im, hi[0][j], lo[0][j]);
        mfma::split_pair<P>(v.im, -v.re, hi[1][j], lo[1][j]);
        mfma::split_pair<P>(w.re, w.im, hi[2][j], lo[2][j]);
        mfma::split_pair<P>(w.im, -w.re, hi[3][j], lo[3][j]);
    }
    uint4* out = frag + ((size_t(r) * gridDim.y + block) * KS + ks) * (SHM_TILES * PARTS * 64) + lane;
#pragma unroll
    for (int i = 0; i < SHM_TILES; i++) {
        out[(i * PARTS) * 64] = uint4 {hi[i][0], hi[i][1], hi[i][2], hi[i][3]};
        if constexpr (LO) out[(i * PARTS + 1) * 64] = uint4 {lo[i][0], lo[i][1], lo[i][2], lo[i][3]};
    }
}

// Partial J^H.y over readouts [r0, r1): partial[chunk][p][v].  Grid (ceil(nv /
// (32 T W)), readout chunks), block 64 W; two fragment buffers of KS 4 PARTS KiB.
template<int T, int W, int KS, bool T8, bool LO>
__global__ void __launch_bounds__(64 * W, W / 4) spiral_hermitian_mfma(
    const SpiralVoxel* __restrict__ voxels, dev::TissueView tissue, const cfloat* __restrict__ m,
    const cfloat* __restrict__ dT1, const cfloat* __restrict__ dT2, const cfloat* __restrict__ dB1,
    const cfloat* __restrict__ dB0, const cfloat* __restrict__ coils, int nc, const uint4* __restrict__ frag,
    int blocks, int groups, const cfloat* __restrict__ k_start, const cfloat* __restrict__ delta_k, int nr, int ns,
    float dt, int r_chunk, cfloat* __restrict__ partial) {
    constexpr int P = LO ? mfma::P_BF16X3 : mfma::P_BF16X1;
    constexpr int S = 8 * KS, NT = T8 ? 8 : 4, NC = T8 ? 2 : 4, PARTS = LO ? 2 : 1;
    constexpr int FRAG = KS * SHM_TILES * PARTS * 64;  // 16-byte words of a block's fragments
    __shared__ uint4 lds[2 * FRAG];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int nv = tissue.nvoxels;
    const int r0 = blockIdx.y * r_chunk, r1 = min(nr, r0 + r_chunk);
    const int vbase = (blockIdx.x * W + wave) * (32 * T);

    int vt[T];
    SpiralVoxel vx[T];
#pragma unroll
    for (int i = 0; i < T; i++) {
        vt[i] = min(vbase + 32 * i + col, nv - 1);
        vx[i] = voxels[vt[i]];
    }
    cfloat g1[T], g2[T], gb1[T], gb0[T], gu[T];
#pragma unroll
    for (int i = 0; i < T; i++) g1[i] = g2[i] = gb1[i] = gb0[i] = gu[i] = {0.0f, 0.0f};

    // a block's fragments, linear in LDS: each wave copies 1 KiB at a time
    auto fetch = [&](int item, int buf) {
        const uint4* from = frag + size_t(item) * FRAG;
#pragma unroll
        for (int k = 0; k < FRAG / 64; k += W) {
            if (FRAG / 64 % W == 0 || k + wave < FRAG / 64) {
                __builtin_amdgcn_global_load_lds(
                    reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(uintptr_t(from + (k + wave) * 64 + lane)),
                    (__attribute__((address_space(3))) uint32_t*)(&lds[buf * FRAG + (k + wave) * 64]), 16, 0, 0);
            }
        }
    };
    int item = r0 * blocks;
    const int last = r1 * blocks;
    int buf = 0;
    if (item < last) fetch(item, 0);

    for (int r = r0; r < r1; r++) {
        const cfloat dk = delta_k[r];
        const double dkx = double(dk.re) / dev::TWO_PI, dky = double(dk.im) / dev::TWO_PI;
        const double k0x = double(k_start[r].re) / dev::TWO_PI;
        cfloat V[T], Vp[T];
#pragma unroll
        for (int i = 0; i < T; i++) V[i] = Vp[i] = {0.0f, 0.0f};
        double turns[T];
        cfloat e1[T], e4[T], e8[T], eS[T];
#pragma unroll
        for (int i = 0; i < T; i++) {
            turns[i] = spiral_turns(vx[i], dkx, dky);
            e1[i] = spiral_phasor(vx[i].decay, turns[i]);
            e4[i] = spiral_phasor(float(4 * half) * vx[i].decay, double(4 * half) * turns[i]);
            e8[i] = spiral_phasor(8.0f * vx[i].decay, 8.0 * turns[i]);
            eS[i] = spiral_phasor(float(S) * vx[i].decay, double(S) * turns[i]);
        }
        for (int block = 0; block < blocks; block++, item++) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of the block's copy
            __syncthreads();                                   // everyone's; and the other buffer has been read
            if (item + 1 < last) fetch(item + 1, buf ^ 1);
            const uint4* a = &lds[buf * FRAG + lane];
            buf ^= 1;

            f32x16 acc[T][SHM_TILES];
#pragma unroll
            for (int i = 0; i < T; i++)
#pragma unroll
                for (int k = 0; k < SHM_TILES; k++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][k][e] = 0.0f;
            cfloat ph[T][4];
#pragma unroll
            for (int i = 0; i < T; i++) {
                ph[i][0] = e4[i];
#pragma unroll
                for (int j = 1; j < 4; j++) ph[i][j] = dev::cmul(ph[i][j - 1], e1[i]);
            }
#pragma unroll 2
            for (int ks = 0; ks < KS; ks++) {
                mfma::bf16x8 bh[T], bl[T];
#pragma unroll
                for (int i = 0; i < T; i++) {
                    uint32_t hw[4], lw[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        mfma::split_pair<P>(ph[i][j].re, ph[i][j].im, hw[j], lw[j]);
                        ph[i][j] = dev::cmul(ph[i][j], e8[i]);
                    }
                    bh[i] = __builtin_bit_cast(mfma::bf16x8, uint4 {hw[0], hw[1], hw[2], hw[3]});
                    bl[i] = __builtin_bit_cast(mfma::bf16x8, uint4 {lw[0], lw[1], lw[2], lw[3]});
                }
#pragma unroll
                for (int k = 0; k < SHM_TILES; k++) {
                    const mfma::bf16x8 ah = __builtin_bit_cast(mfma::bf16x8, a[((ks * SHM_TILES + k) * PARTS) * 64]);
#pragma unroll
                    for (int i = 0; i < T; i++) {
                        acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh[i], acc[i][k], 0, 0, 0);
                        if constexpr (LO) acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl[i], acc[i][k], 0, 0, 0);
                    }
                    if constexpr (LO) {
                        const mfma::bf16x8 al = __builtin_bit_cast(mfma::bf16x8, a[((ks * SHM_TILES + k) * PARTS + 1) * 64]);
#pragma unroll
                        for (int i = 0; i < T; i++)
                            acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh[i], acc[i][k], 0, 0, 0);
                    }
                }
            }

            // sums over t (Horner in conj(E^S)), conj(Phi_sb), the lane's coils
            const int sb = (block / groups) * (S * NT), c0 = (block % groups) * (2 * NC) + NC * half;
#pragma unroll
            for (int i = 0; i < T; i++) {
                const double first = fma(k0x, double(vx[i].x), fma(double(sb), turns[i], -0.5 * double(ns) * vx[i].turns));
                const cfloat phi = spiral_phasor((float(sb) - 0.5f * float(ns)) * vx[i].decay, first);
                cfloat sum = {0.0f, 0.0f}, sump = {0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < NC; k++) {
                    cfloat U, Up;
#pragma unroll
                    for (int t = NT - 1; t >= 0; t--) {
                        const int e = NT * k + t;
                        const cfloat G = {acc[i][0][e], acc[i][1][e]};
                        const cfloat H = {acc[i][2][e], acc[i][3][e]};
                        U = t == NT - 1 ? G : dev::cfma_conj(U, eS[i], G);
                        Up = t == NT - 1 ? H : dev::cfma_conj(Up, eS[i], H);
                    }
                    cfloat C = coils[size_t(min(c0 + k, nc - 1)) * nv + vt[i]];
                    if (c0 + k >= nc) C = {0.0f, 0.0f};
                    sum = dev::cfma_conj(U, C, sum);
                    sump = dev::cfma_conj(Up, C, sump);
                }
                V[i] = dev::cfma_conj(sum, phi, V[i]);
                Vp[i] = dev::cfma_conj(sump, phi, Vp[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < T; i++) {
            const size_t at = size_t(r) * nv + vt[i];
            const cfloat me = m[at], a1 = dT1[at], a2 = dT2[at], ab1 = dB1[at], ab0 = dB0[at];
            const float R2 = 1.0f / vx[i].T2;
            const float kT2 = dt * R2 * R2, kB0 = -dev::TWO_PI_F * dt;
            g1[i] = dev::cfma_conj(V[i], a1, g1[i]);
            g2[i] = dev::cfma_conj(V[i], a2, g2[i]);
            g2[i] = dev::cfma_conj(Vp[i] * kT2, me, g2[i]);
            gb1[i] = dev::cfma_conj(V[i], ab1, gb1[i]);
            gb0[i] = dev::cfma_conj(V[i], ab0, gb0[i]);
            gb0[i] = dev::cfma_conj(cfloat {-Vp[i].im * kB0, Vp[i].re * kB0}, me, gb0[i]);
            gu[i] = dev::cfma_conj(V[i], me, gu[i]);
        }
    }

    // the two halves hold different coils of one voxel
#pragma unroll
    for (int i = 0; i < T; i++) {
        const cfloat rho = tissue.rho(vt[i]);
        cfloat o[5] = {dev::cmul(conj(rho * tissue.T1(vt[i])), g1[i]), dev::cmul(conj(rho * vx[i].T2), g2[i]),
                       dev::cmul(conj(rho), gb1[i]), dev::cmul(conj(rho), gb0[i]), gu[i]};
#pragma unroll
        for (int p = 0; p < 5; p++) {
            o[p].re += __shfl_xor(o[p].re, 32);
            o[p].im += __shfl_xor(o[p].im, 32);
        }
        const int v = vbase + 32 * i + col;
        if (half == 0 && v < nv) {
            cfloat* dst = partial + size_t(blockIdx.y) * 6 * size_t(nv) + v;
#pragma unroll
            for (int p = 0; p < 5; p++) dst[size_t(p) * nv] = o[p];
            dst[size_t(5) * nv] = dev::cmul(o[4], cfloat {0.0f, -1.0f});
        }
    }
}

}  // namespace kernels

bool spiral_hermitian_mfma(
    const CompasContext& ctx, const TissueParameters& p, const cfloat* m, const cfloat* d1, const cfloat* d2,
    const cfloat* db1, const cfloat* db0, const cfloat* coils, int nc, const cfloat* y, const SpiralTrajectory& traj,
    ContractionPrecision precision, cfloat* JHy) {
    if (precision == ContractionPrecision::FP32) return false;
    if (nc > SPIRAL_ADJOINT_COILS) return false;  // the VALU form
    const bool lo = precision == ContractionPrecision::BF16x3 || precision == ContractionPrecision::FP16x3;
    const int nr = traj.nreadouts, ns = traj.samples_per_readout, nv = p.nvoxels;
    // one voxel tile in each of twelve waves, three to a SIMD (at 4 coils x 1120 x
    // 512 over 50176 voxels 5.7 ms; two tiles in each of eight waves spilled, 5.9;
    // sixteen waves 6.3)
    constexpr int T = SPIRAL_ADJOINT_VOXELS / 32, W = SPIRAL_ADJOINT_WAVES;
    const SpiralAdjointLayout l = spiral_adjoint_layout(nv, nr, ns, nc, lo, simd_count(ctx.device()) / 4);
    auto frag = ctx.empty<uint4, 1>({l.fragment_bytes(nr) / int64_t(sizeof(uint4))});
    auto voxels = ctx.empty<kernels::SpiralVoxel, 1>({nv});
    auto partial = ctx.empty<cfloat, 1>({l.partial_bytes(nv) / int64_t(sizeof(cfloat))});
    const auto run = [&](auto ks_c, auto t8_c, auto lo_c) {
        constexpr int KS = decltype(ks_c)::value;
        constexpr bool T8 = decltype(t8_c)::value, LO = decltype(lo_c)::value;
        {
            KernelScope scope(ctx, "spiral_y_fragments");
            const dim3 grid(nr + int(dev::div_ceil(nv, 64 * KS)), l.blocks);
            kernels::spiral_y_fragments<KS, T8, LO><<<grid, 64 * KS, 0, ctx.stream()>>>(
                y, nc, nr, ns, l.groups, frag.data(), dev::tissue_view(p), traj.delta_t, voxels.data());
            check_launch("spiral_y_fragments");
        }
        KernelScope scope(ctx, "spiral_hermitian_mfma");
        kernels::spiral_hermitian_mfma<T, W, KS, T8, LO><<<dim3(l.vblocks, l.chunks), 64 * W, 0, ctx.stream()>>>(
            voxels.data(), dev::tissue_view(p), m, d1, d2, db1, db0, coils, nc, frag.data(), l.blocks, l.groups,
            traj.k_start.data(), traj.delta_k.data(), nr, ns, traj.delta_t, l.r_chunk, partial.data());
        check_launch("spiral_hermitian_mfma");
    };
    const auto with_lo = [&](auto ks_c, auto t8_c) {
        if (lo) run(ks_c, t8_c, std::true_type {});
        else run(ks_c, t8_c, std::false_type {});
    };
    if (l.ks == 1) with_lo(std::integral_constant<int, 1> {}, std::false_type {});
    else if (l.ks == 2) with_lo(std::integral_constant<int, 2> {}, std::false_type {});
    else if (l.ks == 4) with_lo(std::integral_constant<int, 4> {}, std::false_type {});
    else if (!l.t8) with_lo(std::integral_constant<int, 8> {}, std::false_type {});
    else with_lo(std::integral_constant<int, 8> {}, std::true_type {});
    spiral_hermitian_reduce_partials(ctx, partial.data(), l.chunks, nv, JHy);
    return true;
}

}  // namespace compas
