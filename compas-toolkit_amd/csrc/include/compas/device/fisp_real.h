#pragma once
// The FISP EPG recursion of a train whose RF pulses all lie on one axis, in
// real numbers, with or without its forward-mode tangents.
//
// Two facts take the imaginary parts out of the recursion of fisp_epg.h:
//   * Off-resonance.  A spin that precesses by psi = 2 pi B0 TR per TR while
//     the gradient dephases it by theta sees theta + psi, so the state of
//     order k is that of the same voxel on resonance times e^{i k psi}: the
//     rotation mixes F+_k, conj(F-_k) and Z_k, which carry the same factor,
//     the dephasing shift moves F from order k to k + 1 as it gains e^{i psi},
//     and dropping orders >= N does not mix orders.  The echo is F+_0 after
//     another e^{i 2 pi B0 TE}, and that is all that B0 does; its derivative
//     with respect to B0 is i 2 pi TE times the echo.  (Spoiling between
//     repetitions, or the inversion that begins one, clears the transverse
//     states, so the waiting time adds no phase; a train with neither and
//     more than one repetition is not taken here.)
//   * Real pulses.  About +-x the rotation keeps F+ = -i p, F- = i q, Z = z
//     real: with S = p + q and D = p - q,
//       S' = cos(a) S + 2 sin(a) z,  D' = D,  z' = cos(a) z - sin(a) S / 2,
//     a signed.  With decay that is 8 operations per state and TR where the
//     complex form takes 26.
// Both are exact, so this is the same recursion with less rounding (the
// off-resonance phase is applied once, not once per TR).

#include "compas/device/common.h"
#include "compas/device/fisp_common.h"
#include "compas/device/tangent_set.h"

namespace compas {
namespace kernels {

// Whether the launch's train is taken by this form (else fisp_epg_voxel's): the
// RF table ends in an entry that says whether every pulse is real.
__device__ inline bool fisp_real_train(const FispArgs& a) {
    return a.table[a.nslices * a.nTR].w != 0.0f && (a.wait_spoiling || a.inversion || a.repetitions == 1);
}

// v of the lane below (above) in its row of 16 lanes
__device__ __forceinline__ float from_lane_below(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x111, 0xF, 0xF, true));  // row_shr:1
}
__device__ __forceinline__ float from_lane_above(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x101, 0xF, 0xF, true));  // row_shl:1
}

// One TR's coefficients
struct RealTurn {
    float ca, sa, w;       // cos and sin of the signed flip angle; d angle / d B1
    float k1, k2, k3, k4;  // E2 ca / 2, E2 sa, E1 ca, -E1 sa / 2
    float n1, n2, n3, n4;  // their derivatives with respect to B1 (when asked)
};

// The recursion of one voxel (lane `sub` of its LPV <= 16 lanes) over every
// slice profile and repetition.  MASK: the planes written (TangentSet); FORM,
// SIMPLE: as in fisp_epg_voxel_form.  N > (SPL - 1) LPV, so the top state is
// among the last LPV of its lane's.
template<int SPL, int LPV, int MASK, int FORM, bool SIMPLE>
__device__ __forceinline__ void fisp_real_voxel_form(const FispArgs& a, const FispPlanes& out, int voxel, int sub) {
    using TS = TangentSet<MASK & ~TM_B0>;  // B0 needs no states
    constexpr bool B0T = (MASK & TM_B0) != 0;
    constexpr int NT = TS::nt, NP = TangentSet<MASK>::planes, OFS = int(TS::echo);

    const float T1 = a.tissue.T1(voxel);
    const float T2 = a.tissue.T2(voxel);
    const float B1 = a.tissue.B1(voxel);

    const float E1_TE = relax(a.TE, T1), E2_TE = relax(a.TE, T2);
    const float E1_TI = relax(a.TI, T1);
    const float E1_TRmTE = relax(a.TR - a.TE, T1), E2_TRmTE = relax(a.TR - a.TE, T2);
    const float E1_W = relax(a.TW, T1);
    const float E1 = E1_TE * E1_TRmTE, E2 = E2_TE * E2_TRmTE;
    const float hE1 = -0.5f * E1, hE2 = 0.5f * E2;
    // regrowth of Z_0 accumulated over TE and TR-TE
    const float G = E1_TRmTE * (1.0f - E1_TE) + (1.0f - E1_TRmTE);
    // echo = F+_0 E2(TE) e^{i 2 pi B0 TE} with F+_0 = -i p
    const cfloat off = off_resonance(a.TE, a.tissue.B0(voxel));
    const cfloat to_echo = {E2_TE * off.im, -E2_TE * off.re};

    // derivative factors (d/dT of exp(-t/T) = (t/T^2) exp(-t/T))
    const float iT1s = 1.0f / (T1 * T1), iT2s = 1.0f / (T2 * T2);
    const float dE1_TE = a.TE * iT1s * E1_TE, dE1_TRmTE = (a.TR - a.TE) * iT1s * E1_TRmTE;
    const float dE1_TI = a.TI * iT1s * E1_TI, dE1_W = a.TW * iT1s * E1_W;
    const float dG = dE1_TRmTE * (1.0f - E1_TE) - E1_TRmTE * dE1_TE - dE1_TRmTE;
    const float lTR = a.TR * iT1s, k2TR = a.TR * iT2s, k2TE = a.TE * iT2s;
    const float k0TE = dev::TWO_PI_F * a.TE;

    const bool owns_zero = (LPV == 1) || sub == 0;
    const int top = a.N - 1 - sub * SPL;  // the top state's index in this lane, if it is here

    auto turn = [&](float4 t) {
        RealTurn r;
        const float w = t.x * t.y;  // signed flip angle per unit B1
        const float alpha = w * B1;
        float sx, cx;
        half_angle_sincos<FORM>(0.5f * alpha, &sx, &cx);
        r.w = w;
        r.sa = 2.0f * sx * cx;
        r.ca = fmaf(-2.0f * sx, sx, 1.0f);
        r.k1 = hE2 * r.ca;
        r.k2 = E2 * r.sa;
        r.k3 = E1 * r.ca;
        r.k4 = hE1 * r.sa;
        if constexpr (TS::b1) {
            r.n1 = -hE2 * r.sa * w;
            r.n2 = E2 * r.ca * w;
            r.n3 = -E1 * r.sa * w;
            r.n4 = hE1 * r.ca * w;
        }
        return r;
    };

    for (int slice = 0; slice < a.nslices; slice++) {
        const float4* tab = a.table + size_t(slice) * size_t(a.nTR);
        // vector 0 is the state, vectors 1.. its tangents
        float P[1 + NT][SPL], Q[1 + NT][SPL], Z[1 + NT][SPL];
#pragma unroll
        for (int k = 0; k <= NT; k++)
#pragma unroll
            for (int i = 0; i < SPL; i++) P[k][i] = Q[k][i] = Z[k][i] = 0.0f;
        if (owns_zero) Z[0][0] = 1.0f;

        for (int rep = 0; rep < a.repetitions; rep++) {
            const bool sample = (rep == a.repetitions - 1);
            if (rep > 0) {  // spoiled before the waiting time, or by the inversion after it
#pragma unroll
                for (int k = 0; k <= NT; k++)
#pragma unroll
                    for (int i = 0; i < SPL; i++) P[k][i] = Q[k][i] = 0.0f;
#pragma unroll
                for (int i = 0; i < SPL; i++) {
#pragma unroll
                    for (int k = 1; k <= NT; k++) {
                        Z[k][i] *= E1_W;
                        if (TS::t1 && k == 1 + TS::it1) Z[k][i] = fmaf(Z[0][i], dE1_W, Z[k][i]);
                    }
                    Z[0][i] *= E1_W;
                }
                if (owns_zero) {
                    Z[0][0] += 1.0f - E1_W;
                    if constexpr (TS::t1) Z[1 + TS::it1][0] -= dE1_W;
                }
            }
            if (a.inversion) {  // invert (ignores B1), decay(TI), regrow
#pragma unroll
                for (int i = 0; i < SPL; i++) {
#pragma unroll
                    for (int k = 1; k <= NT; k++) {
                        Z[k][i] *= -E1_TI;
                        if (TS::t1 && k == 1 + TS::it1) Z[k][i] = fmaf(-dE1_TI, Z[0][i], Z[k][i]);
                    }
                    Z[0][i] *= -E1_TI;
                }
                if (owns_zero) {
                    Z[0][0] += 1.0f - E1_TI;
                    if constexpr (TS::t1) Z[1 + TS::it1][0] -= dE1_TI;
                }
            }

            // the coefficients of a TR are formed beside the states' update of
            // the TR before it, from a table entry loaded one TR earlier still
            // (the table holds two entries more than the TRs of all slices)
            RealTurn c {}, c_next = turn(tab[0]);
            float4 t_next = tab[1];
            cfloat* rows[NP];
#pragma unroll
            for (int k = 0; k < NP; k++) rows[k] = out.p[k];
            const uint32_t voff = uint32_t(voxel) * uint32_t(sizeof(cfloat));
            for (int n = 0; n < a.nTR; n++) {
                c = c_next;
                const float4 t = t_next;
                t_next = tab[n + 2];
                c_next = turn(t);

                // F+_0 after the pulse (order 0 has p = q), and its tangents over TE
                if ((SIMPLE || sample) && owns_zero) {
                    const float e = fmaf(c.sa, Z[0][0], c.ca * P[0][0]);
                    const cfloat echo = {e * to_echo.re, e * to_echo.im};
                    cfloat v[NP];
                    if constexpr (TS::echo) v[0] = echo;
#pragma unroll
                    for (int k = 0; k < NT; k++) {
                        float d = fmaf(c.sa, Z[1 + k][0], c.ca * P[1 + k][0]);
                        if (TS::t2 && k == TS::it2) d = fmaf(k2TE, e, d);
                        if (TS::b1 && k == TS::ib1) d = fmaf(c.w, fmaf(c.ca, Z[0][0], -c.sa * P[0][0]), d);
                        v[OFS + k] = {d * to_echo.re, d * to_echo.im};
                    }
                    if constexpr (B0T) v[OFS + NT] = {-k0TE * echo.im, k0TE * echo.re};
                    if constexpr (SIMPLE) {
#pragma unroll
                        for (int k = 0; k < NP; k++) {
                            if (k == 0 && NP > 1 && OFS && out.p[0] == nullptr) continue;  // echoes not asked for
                            *reinterpret_cast<cfloat*>(reinterpret_cast<char*>(rows[k]) + voff) = v[k];
                        }
                    } else {
                        for (int u = 0; u < a.usf; u++) {
                            const size_t at = size_t(n * a.usf + u) * size_t(a.tissue.nvoxels) + voxel;
#pragma unroll
                            for (int k = 0; k < NP; k++) {
                                if (k == 0 && NP > 1 && OFS && out.p[0] == nullptr) continue;
                                out.p[k][at] = (slice == 0) ? v[k] : (out.p[k][at] + v[k]);
                            }
                        }
                    }
                }
                if constexpr (SIMPLE) {
#pragma unroll
                    for (int k = 0; k < NP; k++) rows[k] += a.tissue.nvoxels;
                }

                // from the top state down, each state's outputs into their
                // dephased slots after the values there have been read
                float p_top[1 + NT], q_bottom[1 + NT], S[1 + NT], D[1 + NT];
                auto sums = [&](int k, int i, float& Si, float& Di) {
                    if (LPV == 1 && i == SPL - 1 && SPL > 1) {  // F-_{N-1} = 0
                        Si = P[k][i];
                        Di = P[k][i];
                    } else {
                        Si = P[k][i] + Q[k][i];
                        Di = P[k][i] - Q[k][i];
                    }
                };
#pragma unroll
                for (int k = 0; k <= NT; k++) sums(k, SPL - 1, S[k], D[k]);
#pragma unroll
                for (int i = SPL - 1; i >= 0; i--) {
                    float Sn[1 + NT], Dn[1 + NT], pn[1 + NT], qn[1 + NT], zn[1 + NT];
#pragma unroll
                    for (int k = 0; k <= NT; k++) {
                        if (i > 0) sums(k, i - 1, Sn[k], Dn[k]);
                        float u = fmaf(c.k1, S[k], c.k2 * Z[k][i]);
                        float z = fmaf(c.k4, S[k], c.k3 * Z[k][i]);
                        if (TS::b1 && k == 1 + TS::ib1) {
                            u = fmaf(c.n1, S[0], fmaf(c.n2, Z[0][i], u));
                            z = fmaf(c.n4, S[0], fmaf(c.n3, Z[0][i], z));
                        }
                        pn[k] = fmaf(hE2, D[k], u);
                        qn[k] = fmaf(-hE2, D[k], u);
                        if (TS::t2 && k == 1 + TS::it2) {
                            pn[k] = fmaf(k2TR, pn[0], pn[k]);
                            qn[k] = fmaf(k2TR, qn[0], qn[k]);
                        }
                        if (TS::t1 && k == 1 + TS::it1) z = fmaf(lTR, zn[0], z);
                        zn[k] = z;
                    }
#pragma unroll
                    for (int k = 0; k <= NT; k++) {
                        if (i + 1 < SPL) {
                            P[k][i + 1] = pn[k];  // dephasing: F+_{i+1} <- F+_i
                        } else {
                            p_top[k] = pn[k];
                        }
                        if (i > 0) {
                            Q[k][i - 1] = qn[k];  // dephasing: F-_{i-1} <- F-_i
                        } else {
                            q_bottom[k] = qn[k];
                        }
                        Z[k][i] = zn[k];
                        S[k] = Sn[k];
                        D[k] = Dn[k];
                    }
                }
                if (owns_zero) {
                    Z[0][0] += G;
                    if constexpr (TS::t1) Z[1 + TS::it1][0] += dG;
                }
                // the ends of the dephasing: neighbouring lanes, F-_{N-1} <- 0 (what
                // lies above it never comes back down), F+_0 <- conj(F-_0)
#pragma unroll
                for (int k = 0; k <= NT; k++) {
                    if constexpr (LPV > 1) {
                        P[k][0] = from_lane_below(p_top[k]);
                        Q[k][SPL - 1] = from_lane_above(q_bottom[k]);
#pragma unroll
                        for (int i = SPL > LPV ? SPL - LPV : 0; i < SPL; i++)
                            if (i == top) Q[k][i] = 0.0f;
                    } else {
                        Q[k][SPL - 1] = 0.0f;
                    }
                    if (owns_zero) P[k][0] = Q[k][0];
                }
            }
        }
    }
}

// fisp_real_voxel_form in the form the wave needs, as fisp_epg_voxel chooses.
// A pass of several fields may leave out its first plane, the echoes.
template<int SPL, int LPV, int MASK>
__device__ __forceinline__ void fisp_real_voxel(const FispArgs& a, const FispPlanes& out, int voxel, int sub) {
    const FispWaveForm f = fisp_wave_form(a, voxel);
    if constexpr (MASK == TM_ECHO) {
        if (f.wide) {
            fisp_real_voxel_form<SPL, LPV, MASK, HALF_WIDE, false>(a, out, voxel, sub);
        } else if (!f.plain) {
            fisp_real_voxel_form<SPL, LPV, MASK, HALF_POLY, false>(a, out, voxel, sub);
        } else if (!f.q0) {
            fisp_real_voxel_form<SPL, LPV, MASK, HALF_POLY, true>(a, out, voxel, sub);
        } else {
            fisp_real_voxel_form<SPL, LPV, MASK, HALF_Q0, true>(a, out, voxel, sub);
        }
    } else if (f.wide || !f.plain) {  // two forms only: there are many tangent kernels
        fisp_real_voxel_form<SPL, LPV, MASK, HALF_WIDE, false>(a, out, voxel, sub);
    } else {
        fisp_real_voxel_form<SPL, LPV, MASK, HALF_POLY, true>(a, out, voxel, sub);
    }
}

}  // namespace kernels
}  // namespace compas
