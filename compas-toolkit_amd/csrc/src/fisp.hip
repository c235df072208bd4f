// FISP extended-phase-graph simulation on gfx950.
//
// Semantics: reference src/simulate/fisp_kernels.cuh:99-244, fisp.cu:7-140 and
// the EPG operators of src/operators/epg.cuh:19-322 (see the oracle for the
// literal restatement).
//
// A train of real pulses takes the real recursion (fisp_real.h); both kernels
// are launched and one leaves at once.
//
// Design of the complex form (MI355X):
//   * One voxel per lane (or LPV lanes per voxel for large state counts or
//     small voxel counts).  The F+/F-/Z states of a voxel live in VGPRs; the
//     dephasing shift is a register rename inside the unrolled update.
//   * The per-TR operator "excite -> decay(TE) -> regrow -> decay(TR-TE) ->
//     regrow" is one real 3x3 matrix M = D(TR) R(alpha, phi) acting on the
//     state written in the real transverse basis X = (F+ + F-)/2,
//     Y = (F+ - F-)/(2i): 18 FMAs per state instead of ~40 for the complex
//     F+/F-/Z form; the basis change costs 8 adds.  The TE sample F+_0(TE) is
//     the updated state 0 over the decay after TE (fisp_direct_echo: from the
//     first two rows of D(TE) R where that decay underflows).
//   * The RF table (alpha per unit B1, cos phi, sin phi) is precomputed per
//     (slice, TR) and read with wave-uniform (scalar) loads.
//   * Echoes are written directly in [nreadouts][nvoxels] layout (coalesced
//     over voxels), including the undersampling expansion, so no transpose
//     pass is needed.

#include <cfloat>
#include <algorithm>
#include <cmath>

#include <cstdlib>
#include <mutex>
#include <sstream>

#include "compas/device/common.h"
#include "compas/device/fisp_common.h"
#include "compas/device/fisp_launch.h"
#include "compas/internal.h"

namespace compas {
namespace kernels {

// The RF table (FispArgs::table) with its two closing entries.  One workgroup
// of 1024 threads: every wave of the recursion needs the train's largest flip
// angle and whether its pulses are real, and would otherwise look through the
// whole table for them.
__global__ void __launch_bounds__(1024) fisp_rf_table(
    const cfloat* RF, const cfloat* profiles, int nTR, int nslices, float4* table) {
    __shared__ float s_max[16];
    __shared__ int s_real;
    const int total = nTR * nslices;
    if (threadIdx.x == 0) s_real = 1;
    __syncthreads();
    float largest = 0.0f;
    bool real = true;
    for (int i = threadIdx.x; i < total; i += 1024) {
        const cfloat p = profiles[i], r = RF[i % nTR];
        const cfloat rf = {p.re * r.re - p.im * r.im, p.re * r.im + p.im * r.re};
        const float a = hypotf(rf.re, rf.im);
        float c = 1.0f, s = 0.0f;
        if (a > FLT_MIN) {  // epg.cuh:64-67
            c = rf.re / a;
            s = rf.im / a;
        }
        table[i] = make_float4(dev::DEG2RAD_F * a, c, s, 0.0f);
        largest = fmaxf(largest, dev::DEG2RAD_F * a);
        real = real && s == 0.0f;
    }
    for (int off = 32; off > 0; off >>= 1) largest = fmaxf(largest, __shfl_xor(largest, off));
    if (threadIdx.x % 64 == 0) s_max[threadIdx.x / 64] = largest;
    if (!real) s_real = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) largest = fmaxf(largest, s_max[w]);
        table[total] = make_float4(largest, 0.0f, 0.0f, s_real ? 1.0f : 0.0f);
        table[total + 1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

}  // namespace kernels

Array<float4, 1> fisp_rf_table(const CompasContext& ctx, const FISPSequence& seq) {
    const int nTR = int(seq.RF_train.size(0)), nslices = int(seq.sliceprofiles.size(0));
    auto table = ctx.empty<float4, 1>({int64_t(nslices) * nTR + 2});
    KernelScope ks(ctx, "fisp_rf_table");
    kernels::fisp_rf_table<<<1, 1024, 0, ctx.stream()>>>(
        seq.RF_train.data(), seq.sliceprofiles.data(), nTR, nslices, table.data());
    check_launch("fisp_rf_table");
    return table;
}

int simd_count(int device) {
    static int cached[64] = {0};
    if (device >= 0 && device < 64 && cached[device]) return cached[device];
    hipDeviceProp_t prop;
    COMPAS_HIP_CHECK(hipGetDeviceProperties(&prop, device));
    int n = prop.multiProcessorCount * 4;  // 4 SIMDs per CU on CDNA
    if (device >= 0 && device < 64) cached[device] = n;
    return n;
}

// Lanes per voxel and states per lane of the complex form: the lowest modelled
// time of a TR, in us, of k = ceil(waves / SIMDs) waves sharing a SIMD with s
// states per lane.  A wave alone is bound by its chain of operations, which a
// second one fits beside; from then on the instructions issued count, and an
// odd wave costs nearly a pair.  Measured and modelled, in 1, 2, 4 and 8 lanes:
// 28701 voxels x 16 states 0.93 0.93, 0.58 0.58, 0.45 0.46, 0.62 0.61; 50176 x
// 25 1.35 1.32, 0.88 0.87, 1.13 1.15, 1.39 1.56; 20011 x 37 -, 1.13 1.06, 0.79
// 0.74, 0.87 0.93; 200000 x 25 3.21 3.10, 3.38 3.65.  With 37 states 20011 voxels
// take 0.79 in four lanes of ten (1.79 in two of 32, the only layout before for
// 33 to 64 states), 5000 x 60 0.62 in eight (1.72).
static void choose_fisp_layout(int N, int nvoxels, int simds, int* spl, int* lpv) {
    double best = 1e300;
    for (int l : {1, 2, 4, 8}) {
        const int s = (N + l - 1) / l;
        if (!fisp_epg_launcher(l, s)) continue;
        double k = std::ceil(double(nvoxels) * l / 64.0 / simds);
        if (k > 2.0) k = 2.0 * std::ceil(0.5 * k);
        const double cost = std::max(0.24 + 0.043 * s, 0.15 + 0.06 * k + s * (0.031 * k - 0.0155));
        if (cost < best) {
            best = cost;
            *spl = s;
            *lpv = l;
        }
    }
}

static void check_fisp_sequence(const FISPSequence& seq) {
    COMPAS_CHECK(seq.max_state >= 1);
    if (seq.max_state > 128) COMPAS_ERROR("max_state cannot exceed 128");  // fisp.cu:100-102
    COMPAS_CHECK(seq.sliceprofiles.size(1) == seq.RF_train.size(0));  // fisp.cu:22
    COMPAS_CHECK(seq.undersampling_factor >= 1);
    COMPAS_CHECK(seq.repetitions >= 1);
}

// Launches the recursion for every voxel: `table` holds the RF table of
// `seq` (fisp_rf_table), `echos` the [nTR * usf][nvoxels] output.
static void launch_fisp_epg(
    const CompasContext& ctx, const TissueParameters& parameters, const FISPSequence& seq, const float4* table,
    cfloat* echos, bool timed);

Array<cfloat, 2> simulate_magnetization(
    const CompasContext& ctx,
    TissueParameters parameters,
    FISPSequence seq) {
    check_fisp_sequence(seq);
    const int nTR = int(seq.RF_train.size(0));
    const int nv = parameters.nvoxels;
    const int nslices = int(seq.sliceprofiles.size(0));
    const int nr = nTR * seq.undersampling_factor;
    ctx.activate();

    auto echos = ctx.empty<cfloat, 2>({nr, nv});
    if (nv == 0 || nr == 0) return echos;
    if (nslices == 0) {
        ctx.fill_zero(echos.data(), echos.nbytes());
        return echos;
    }

    auto table = fisp_rf_table(ctx, seq);
    launch_fisp_epg(ctx, parameters, seq, table.data(), echos.data(), true);
    return echos;
}

// ---------------------------------------------------------------------------
// Allocation-free variant: the RF table lives in a file-scope device array
// instead of the context's pool, and the caller provides the echo buffer.
//
// Each GPU holds its own copy of `scratch` for the life of the process.  In
// host code the name `scratch` is a host-side stand-in, never a device
// address: the per-device address comes from hipGetSymbolAddress, looked up
// once per device with that device current, and only that address is passed
// to kernels.  Calls on one GPU share the array, so calls that overlap on one
// GPU (different streams or threads without ordering) race; calls on one
// context's stream are ordered and safe.

static constexpr int64_t kRfTableScratchEntries = int64_t(1) << 16;  // (slice, TR) pairs: 1 MiB

static __device__ __align__(256) float4 scratch[kRfTableScratchEntries + 2];  // and the two closing entries

static float4* scratch_address(int device) {
    static std::mutex mutex;
    static float4* address[256] = {};
    if (device < 0 || device >= 256) COMPAS_ERROR("device ordinal out of range");
    std::lock_guard<std::mutex> lock(mutex);
    if (address[device] == nullptr) {
        void* p = nullptr;
        COMPAS_HIP_CHECK(hipSetDevice(device));
        COMPAS_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) COMPAS_ERROR("no device address for the RF-table scratch array");
        address[device] = static_cast<float4*>(p);
    }
    return address[device];
}

void simulate_magnetization_into(
    const CompasContext& ctx, const TissueParameters& parameters, const FISPSequence& seq, cfloat* echos,
    int64_t capacity) {
    check_fisp_sequence(seq);
    const int64_t nTR = seq.RF_train.size(0);
    const int64_t nv = parameters.nvoxels;
    const int64_t nslices = seq.sliceprofiles.size(0);
    const int64_t nr = nTR * seq.undersampling_factor;
    if (nslices * nTR > kRfTableScratchEntries) {
        std::stringstream ss;
        ss << "sequence too large for the allocation-free FISP simulation: " << nslices << " slice profiles x " << nTR
           << " TRs = " << nslices * nTR << " RF-table entries, at most " << kRfTableScratchEntries;
        throw CompasException(ss.str());
    }
    if (capacity < nr * nv) {
        std::stringstream ss;
        ss << "echo buffer too small: " << capacity << " complex values for [" << nr << "][" << nv << "]";
        throw CompasException(ss.str());
    }
    if (nr * nv == 0) return;
    if (echos == nullptr) COMPAS_ERROR("null echo buffer");
    ctx.activate();
    if (nslices == 0) {
        ctx.fill_zero(echos, size_t(nr * nv) * sizeof(cfloat));
        return;
    }
    float4* table = scratch_address(ctx.device());
    kernels::fisp_rf_table<<<1, 1024, 0, ctx.stream()>>>(
        seq.RF_train.data(), seq.sliceprofiles.data(), int(nTR), int(nslices), table);
    check_launch("fisp_rf_table");
    launch_fisp_epg(ctx, parameters, seq, table, echos, false);
}

static void launch_fisp_epg(
    const CompasContext& ctx, const TissueParameters& parameters, const FISPSequence& seq, const float4* table,
    cfloat* echos, bool timed) {
    const int nTR = int(seq.RF_train.size(0));
    const int nv = parameters.nvoxels;
    const int nslices = int(seq.sliceprofiles.size(0));

    kernels::FispArgs a;
    a.tissue = dev::tissue_view(parameters);
    a.table = table;
    a.nTR = nTR;
    a.nslices = nslices;
    a.TR = seq.TR;
    a.TE = seq.TE;
    a.TW = seq.TW;
    a.TI = seq.TI;
    a.N = seq.max_state;
    a.usf = seq.undersampling_factor;
    a.repetitions = seq.repetitions;
    a.inversion = seq.inversion_prepulse;
    a.wait_spoiling = seq.wait_spoiling;
    a.echos = echos;

    int spl = 0, lpv = 0;
    choose_fisp_layout(seq.max_state, nv, simd_count(ctx.device()), &spl, &lpv);
    if (const char* e = std::getenv("COMPAS_FISP_LPV")) {  // layout override (1, 2, 4 or 8 lanes per voxel)
        const int l = std::atoi(e);
        const int s = l > 0 ? (seq.max_state + l - 1) / l : 0;
        if (fisp_epg_launcher(l, s)) {
            spl = s;
            lpv = l;
        }
    }
    const FispLauncher fn = fisp_epg_launcher(lpv, spl);
    COMPAS_CHECK(fn != nullptr);
    unsigned blocks = dev::div_ceil(int64_t(nv) * lpv, 64);
    // both forms are launched, and the one that does not suit the train leaves
    // at once: what the train is like is known on the device only
    const auto launch = [&] {
        launch_fisp_real(ctx, a, kernels::TM_ECHO, kernels::FispPlanes {{echos}});
        fn(a, blocks, ctx.stream());
        check_launch("fisp_epg");
    };
    if (timed) {
        KernelScope ks(ctx, "fisp_epg");
        launch();
    } else {
        launch();
    }
}

}  // namespace compas
