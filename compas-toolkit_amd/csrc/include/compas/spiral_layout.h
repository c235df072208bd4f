#pragma once
// Layout of the spiral J^H.y on MFMA (jacobian_spiral_mfma.hip), shared with the
// request server's memory estimate.  Host code only.

#include <algorithm>
#include <cstdint>

namespace compas {

constexpr int SPIRAL_ADJOINT_COILS = 8;    // more coils take the VALU form
constexpr int SPIRAL_ADJOINT_WAVES = 12;   // waves of a workgroup, three to a SIMD: one workgroup to a CU
constexpr int SPIRAL_ADJOINT_VOXELS = 32;  // voxels of a wave

struct SpiralAdjointLayout {
    int ks;               // K steps of a sample block: S = 8 ks
    bool t8;              // eight t of four coils to a row tile, else four t of eight
    int groups, blocks;   // coil groups; blocks (sample block x coil group) of a readout
    int64_t words;        // 16-byte words of a block's operand fragments
    int vblocks;          // workgroups over the voxels
    int r_chunk, chunks;  // readouts summed in FP32 by one workgroup, and how many such ranges
    int64_t fragment_bytes(int nr) const { return int64_t(nr) * blocks * words * 16; }
    int64_t partial_bytes(int nv) const { return int64_t(chunks) * 6 * nv * 8; }
};

// nv, nr, ns >= 1, 1 <= nc <= SPIRAL_ADJOINT_COILS; lo: hi + lo operands; slots:
// resident workgroups
inline SpiralAdjointLayout spiral_adjoint_layout(int nv, int nr, int ns, int nc, bool lo, int slots) {
    const auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    SpiralAdjointLayout l;
    // four t of the smallest S that holds the samples, eight t of S = 64 for more
    // than 256, blocks of 512 beyond
    l.ks = ns <= 32 ? 1 : ns <= 64 ? 2 : ns <= 128 ? 4 : 8;
    l.t8 = ns > 256;
    l.groups = int(up(nc, l.t8 ? 4 : 8));
    l.blocks = l.groups * int(up(ns, 8 * l.ks * (l.t8 ? 8 : 4)));
    l.words = int64_t(l.ks) * 4 * (lo ? 2 : 1) * 64;  // four row tiles of 64 lanes
    l.vblocks = int(up(nv, SPIRAL_ADJOINT_VOXELS * SPIRAL_ADJOINT_WAVES));
    // readout chunks: the fewest rounds of resident workgroups times a chunk's
    // readouts (and two readouts' worth of beginning and end).  A chunk is summed
    // in FP32 and the chunks in FP64, so a chunk is no longer than 192 readouts
    // (98304 voxels x 1120 readouts in one chunk: 4.9e-7 of a constant sum, in six
    // 8e-8)
    l.r_chunk = nr;
    int64_t best = INT64_MAX;
    const int fewest = int(up(nr, 192));
    for (int n = fewest; n <= nr && (n == fewest || int64_t(n) * l.vblocks <= 8 * int64_t(slots)); n++) {
        const int size = int(up(nr, n));
        const int64_t cost = up(up(nr, size) * l.vblocks, slots) * (size + 2);
        if (cost < best) {
            best = cost;
            l.r_chunk = size;
        }
    }
    l.chunks = int(up(nr, l.r_chunk));
    return l;
}

}  // namespace compas
