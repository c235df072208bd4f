// Spiral sums out[c][r][s] = sum_v C[c][v] (A[r][v] + (s - ns/2) Ab[r][v]) E_rv^s
// (signal: A only; J.v: both amplitudes) with the voxel sum on MFMA (BF16 hi +
// lo, or hi only; FP32 accumulation).
//
// With s = sb + S t + n, S = 32 CT, E^s = E^(sb + S t) E^n, so a readout's sum
// is a complex GEMM with rows (coil, t), columns n < S and K = voxels: A = C A_r
// E^(sb + S t), B = E^n.  Per voxel and readout nc T + S elements are generated
// instead of one for every sample (96 instead of 512 at 4 coils x 512
// samples), for the same MFMA products.  Of two amplitudes each has rows of its
// own; the pass that adds the voxel ranges multiplies the second sum by s - ns/2
// (taken apart into sb + S t - ns/2 and n, its two terms would cancel near the
// centre of the readout after each was rounded).
//
// A wave owns a readout and a voxel range and walks it eight voxels at a time
// (one K step of v_mfma_f32_32x32x16_bf16):
//   * generate: lane (voxel l % 8, slot q = l / 8) forms E^q and E^(sb + S q),
//     one phasor each, steps through E^(q + 8 m) with E^8 = (E^4)^2 from a
//     neighbouring lane, splits them and leaves B's hi and lo words and A_r
//     E^(sb + S q) in LDS;
//   * contract: lane l reads B's column l % 32 and, for its row (coil, t), four
//     voxels' amplitudes, multiplies them with the coil map, and splits the rows
//     of the real and of the imaginary part, (w_re, -w_im) and (w_im, w_re).
// Rows: T is a power of two up to 8, row = coil T + t, 32 to a tile, RT tiles
// (coils beyond nc and samples beyond ns are computed and not stored); 32 RT CT
// accumulator registers.  Voxel ranges of one readout are summed by a second
// pass over the partial planes in FP64 (deterministic).
//
// What bounds it: VALU issue (the splits are a third of it) at the clock that
// the matrix units leave.  At 4 coils x 1120 x 512 over 50176 voxels the signal
// takes 4.1 ms and J.v 6.7 ms with their amplitude passes (13.1 and 13.8 ms
// when every sample's element was generated), VALU busy 77% and MFMA 33% of the
// cycles at 2.1 GHz, with two amplitudes 72% and 43% at 2.0 GHz.  Tried without gain: the next step's generation beside the
// MFMAs (two LDS buffers, with and without scheduling groups), the two
// amplitudes in two waves of a workgroup, four waves per SIMD.
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

namespace compas {
namespace kernels {

__device__ inline mfma::bf16x8 pack_bf16x8(const uint32_t (&w)[4]) {
    const uint4 v = {w[0], w[1], w[2], w[3]};
    return __builtin_bit_cast(mfma::bf16x8, v);
}

// The pairs of w in the rows of the real and of the imaginary part, (w_re,
// -w_im) and (w_im, w_re), split into BF16 hi + lo: the conversions take the
// sign and the order for nothing.
template<bool LO>
__device__ __forceinline__ void split_rows(cfloat w, uint32_t& rh, uint32_t& rl, uint32_t& ih, uint32_t& il) {
    const mfma::bf16x2 h = {(__bf16)w.re, (__bf16)-w.im}, hi = {(__bf16)w.im, (__bf16)w.re};
    rh = __builtin_bit_cast(uint32_t, h);
    ih = __builtin_bit_cast(uint32_t, hi);
    if constexpr (LO) {
        const float re = w.re - __builtin_bit_cast(float, rh << 16), im = w.im - __builtin_bit_cast(float, ih << 16);
        rl = __builtin_bit_cast(uint32_t, mfma::bf16x2 {(__bf16)re, (__bf16)-im});
        il = __builtin_bit_cast(uint32_t, mfma::bf16x2 {(__bf16)im, (__bf16)re});
    } else {
        rl = il = 0u;
    }
}

typedef float f32x16s __attribute__((ext_vector_type(16)));

// grid (nr, voxel ranges, sample passes), block 64
template<int CT, int RT, bool TWO, bool LO>
__global__ void __launch_bounds__(64, 2) spiral_sum_split(
    const SpiralVoxel* __restrict__ voxels, int nv, const cfloat* __restrict__ A, const cfloat* __restrict__ Ab,
    const cfloat* __restrict__ coils, int nc, const cfloat* __restrict__ delta_k, int nr, int ns, int tbits,
    int v_chunk, cfloat* __restrict__ partial) {
    static_assert(!TWO || RT == 2, "the two amplitudes take a row tile each");
    constexpr int P = LO ? mfma::P_BF16X3 : mfma::P_BF16X1;
    constexpr int S = 32 * CT;
    __shared__ __align__(16) uint32_t b_hi[S * 8], b_lo[LO ? S * 8 : 4];
    __shared__ __align__(16) float2 amp[TWO ? 2 : 1][8 * 8];
    const int lane = threadIdx.x;
    const int gv = lane & 7, q = lane >> 3;      // generating: voxel of the step, slot
    const int col = lane & 31, half = lane >> 5;  // contracting: row / column, half of the voxels
    const int r = blockIdx.x;
    const int v_begin = blockIdx.y * v_chunk, v_end = min(nv, v_begin + v_chunk);
    const int sb = blockIdx.z * (S << tbits);
    const int t = col & ((1 << tbits) - 1);
    const size_t row = size_t(r) * nv;
    const cfloat dk = delta_k[r];
    const double dkx = double(dk.re) / dev::TWO_PI, dky = double(dk.im) / dev::TWO_PI;
    const cfloat* coil_row[TWO ? 1 : RT];
#pragma unroll
    for (int i = 0; i < (TWO ? 1 : RT); i++) {
        const int c = (col >> tbits) + i * (32 >> tbits);
        coil_row[i] = coils + size_t(min(c, nc - 1)) * nv;
    }

    f32x16s acc[RT][2][CT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int j = 0; j < CT; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][k][j][e] = 0.0f;

    const float s_amp = float(sb + S * q);  // the slot's sample
    // the next step's voxel is loaded a step ahead
    SpiralVoxel nx;
    cfloat na, nb {};
    auto load = [&](int vk) {
        const int v = min(vk + gv, v_end - 1);
        nx = voxels[v];
        na = A[row + v];
        if constexpr (TWO) nb = Ab[row + v];
        if (vk + gv >= v_end) na = nb = {0.0f, 0.0f};
    };
    load(v_begin);
    for (int vk = v_begin; vk < v_end; vk += 8) {
        const SpiralVoxel x = nx;
        const cfloat a = na, ab = nb;
        load(vk + 8);
        cfloat cm[TWO ? 1 : RT][4];
#pragma unroll
        for (int i = 0; i < (TWO ? 1 : RT); i++)
#pragma unroll
            for (int j = 0; j < 4; j++) cm[i][j] = coil_row[i][min(vk + 4 * half + j, nv - 1)];

        const double turns = spiral_turns(x, dkx, dky);
        cfloat ph = spiral_phasor(float(q) * x.decay, double(q) * turns);
        cfloat e8 = {__shfl(ph.re, 32 + gv), __shfl(ph.im, 32 + gv)};
        e8 = dev::cmul(e8, e8);
        const cfloat w = spiral_phasor(s_amp * x.decay, double(s_amp) * turns);
        const cfloat u = dev::cmul(a, w);
        amp[0][lane] = make_float2(u.re, u.im);
        if constexpr (TWO) {
            const cfloat ub = dev::cmul(ab, w);
            amp[1][lane] = make_float2(ub.re, ub.im);
        }
#pragma unroll
        for (int m = 0; m < S / 8; m++) {
            uint32_t h, l;
            mfma::split_pair<P>(ph.re, ph.im, h, l);
            b_hi[64 * m + lane] = h;
            if constexpr (LO) b_lo[64 * m + lane] = l;
            if (m + 1 < S / 8) ph = dev::cmul(ph, e8);
        }
        __syncthreads();  // one wave: orders the LDS accesses

        mfma::bf16x8 bh[CT], bl[CT];
#pragma unroll
        for (int j = 0; j < CT; j++) {
            bh[j] = *reinterpret_cast<const mfma::bf16x8*>(&b_hi[(32 * j + col) * 8 + 4 * half]);
            if constexpr (LO) bl[j] = *reinterpret_cast<const mfma::bf16x8*>(&b_lo[(32 * j + col) * 8 + 4 * half]);
        }
#pragma unroll
        for (int i = 0; i < RT; i++) {
            uint32_t rh[4], rl[4], ih[4], il[4];
            const float4* p = reinterpret_cast<const float4*>(&amp[TWO ? i : 0][8 * t + 4 * half]);
            const float4 p01 = p[0], p23 = p[1];
            const cfloat pv[4] = {{p01.x, p01.y}, {p01.z, p01.w}, {p23.x, p23.y}, {p23.z, p23.w}};
#pragma unroll
            for (int j = 0; j < 4; j++)
                split_rows<LO>(dev::cmul(cm[TWO ? 0 : i][j], pv[j]), rh[j], rl[j], ih[j], il[j]);
            const mfma::bf16x8 ah[2] = {pack_bf16x8(rh), pack_bf16x8(ih)}, al[2] = {pack_bf16x8(rl), pack_bf16x8(il)};
            // one product over all tiles, then the next: no MFMA waits for the one before it
#pragma unroll
            for (int product = 0; product < (LO ? 3 : 1); product++)
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int j = 0; j < CT; j++)
                        acc[i][k][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            product == 2 ? al[k] : ah[k], product == 1 ? bl[j] : bh[j], acc[i][k][j], 0, 0, 0);
        }
        __syncthreads();
    }

    // with two amplitudes a plane for each
    const size_t plane = size_t(nc) * nr * ns;
    cfloat* base = partial + size_t(blockIdx.y) * (TWO ? 2 : 1) * plane;
#pragma unroll
    for (int i = 0; i < (TWO ? 1 : RT); i++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int rho = 32 * i + 8 * (e / 4) + 4 * half + (e % 4);
            const int c = rho >> tbits, tt = rho & ((1 << tbits) - 1);
#pragma unroll
            for (int j = 0; j < CT; j++) {
                const int n = 32 * j + col, s = sb + S * tt + n;
                if (c < nc && s < ns) {
                    const size_t o = (size_t(c) * nr + r) * ns + s;
                    base[o] = {acc[i][0][j][e], acc[i][1][j][e]};
                    if constexpr (TWO) base[plane + o] = {acc[RT - 1][0][j][e], acc[RT - 1][1][j][e]};
                }
            }
        }
}

// out[i] = sum over the splits (FP64, in a fixed order); with two amplitudes out
// = first + (s - ns/2) second, s = i % ns.  `parts` (a power of two up to 64)
// lanes share an output, each a range of its splits.
template<bool TWO>
__global__ void spiral_sum_reduce(
    const cfloat* __restrict__ partial, int splits, int parts, int64_t n, int ns, cfloat* __restrict__ out) {
    for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n * parts; t += int64_t(gridDim.x) * blockDim.x) {
        const int64_t i = t / parts;
        const int part = int(t % parts), per = (splits + parts - 1) / parts;
        double re = 0.0, im = 0.0, bre = 0.0, bim = 0.0;
        for (int k = part * per; k < min(splits, (part + 1) * per); k++) {
            const size_t o = size_t(k) * (TWO ? 2 : 1) * size_t(n) + size_t(i);
            const cfloat p = partial[o];
            re += p.re;
            im += p.im;
            if constexpr (TWO) {
                const cfloat q = partial[o + size_t(n)];
                bre += q.re;
                bim += q.im;
            }
        }
        if constexpr (TWO) {
            const double sp = double(i % ns) - 0.5 * double(ns);
            re = fma(sp, bre, re);
            im = fma(sp, bim, im);
        }
        for (int off = 1; off < parts; off <<= 1) {
            re += __shfl_xor(re, off);
            im += __shfl_xor(im, off);
        }
        if (part == 0) out[i] = {float(re), float(im)};
    }
}

}  // namespace kernels

bool spiral_sum_on_mfma(int nc, bool two, ContractionPrecision precision) {
    return precision != ContractionPrecision::FP32 && nc <= (two ? 4 : 8);  // what the row tiles hold
}

void spiral_sum_mfma(
    const CompasContext& ctx, const kernels::SpiralVoxel* voxels, int nv, const cfloat* A, const cfloat* Ab,
    const cfloat* coils, int nc, const SpiralTrajectory& t, ContractionPrecision precision, cfloat* out) {
    const bool two = Ab != nullptr;
    const bool lo = precision == ContractionPrecision::BF16x3 || precision == ContractionPrecision::FP16x3;
    const int nr = t.nreadouts, ns = t.samples_per_readout;
    // S = 64 columns for more than 256 samples (half as many rows to generate per
    // column), 32 below; up to 8 S samples a pass
    const int ct = ns > 256 ? 2 : 1;
    const int S = 32 * ct;
    int tbits = 0;
    while (tbits < 3 && (S << tbits) < ns) tbits++;
    const int passes = int(dev::div_ceil(ns, S << tbits));
    const int rt = two || (nc << tbits) > 32 ? 2 : 1;
    // voxel splits: about eight waves per SIMD in the grid (two or three are
    // resident; with four, 1.4 rounds of them took 10% longer), sixteen K steps
    // each at least
    const int want = int(std::max<int64_t>(1, dev::div_ceil(8 * 1024, int64_t(nr) * passes)));
    const int splits0 = std::min(want, int(dev::div_ceil(nv, 128)));
    const int v_chunk = int(dev::div_ceil(dev::div_ceil(nv, splits0), 8)) * 8;
    const int splits = int(dev::div_ceil(nv, v_chunk));
    const int64_t plane = int64_t(nc) * nr * ns;
    auto partial = ctx.empty<cfloat, 1>({int64_t(splits) * (two ? 2 : 1) * plane});
    {
        KernelScope ks(ctx, "spiral_sum_mfma");
        const dim3 grid(nr, splits, passes);
        const auto launch = [&](auto ct_c, auto rt_c, auto two_c, auto lo_c) {
            kernels::spiral_sum_split<decltype(ct_c)::value, decltype(rt_c)::value, decltype(two_c)::value, decltype(lo_c)::value>
                <<<grid, 64, 0, ctx.stream()>>>(voxels, nv, A, Ab, coils, nc, t.delta_k.data(), nr, ns, tbits,
                                                v_chunk, partial.data());
        };
        const auto with_lo = [&](auto ct_c, auto rt_c, auto two_c) {
            if (lo) launch(ct_c, rt_c, two_c, std::true_type {});
            else launch(ct_c, rt_c, two_c, std::false_type {});
        };
        const auto with_ct = [&](auto rt_c, auto two_c) {
            if (ct == 2) with_lo(std::integral_constant<int, 2> {}, rt_c, two_c);
            else with_lo(std::integral_constant<int, 1> {}, rt_c, two_c);
        };
        if (two) with_ct(std::integral_constant<int, 2> {}, std::true_type {});
        else if (rt == 2) with_ct(std::integral_constant<int, 2> {}, std::false_type {});
        else with_ct(std::integral_constant<int, 1> {}, std::false_type {});
        check_launch("spiral_sum_mfma");
    }
    KernelScope ks(ctx, "spiral_sum_reduce");
    // a few readouts have few outputs of many splits each: 512 outputs of 2048
    // splits took 250 us (two amplitudes 500) with one lane to an output
    int parts = 1;
    while (parts < 64 && 2 * parts <= splits && plane * parts < (1 << 16)) parts *= 2;
    const unsigned blocks = unsigned(std::min<int64_t>(dev::div_ceil(plane * parts, int64_t(256)), 8192));
    if (two) kernels::spiral_sum_reduce<true><<<blocks, 256, 0, ctx.stream()>>>(partial.data(), splits, parts, plane, ns, out);
    else kernels::spiral_sum_reduce<false><<<blocks, 256, 0, ctx.stream()>>>(partial.data(), splits, parts, plane, ns, out);
    check_launch("spiral_sum_reduce");
}

}  // namespace compas
