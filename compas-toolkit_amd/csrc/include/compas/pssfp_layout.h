#pragma once
// Workgroup layout of the pSSFP kernels that sum over slice positions inside a
// workgroup (pssfp_map.hip, pssfp_map_tangent.hip).  Host code only.

namespace compas {

struct PssfpWorkgroup {
    int nv_block;  // voxels of a workgroup
    int nz_group;  // slice positions of a group; nv_block nz_group <= lanes
    int groups;    // ceil(nz / nz_group)
};

// nz >= 1 slice positions in groups of equal size, at most `most` (<= lanes)
// each, such that the most of the `lanes` isochromats of a workgroup are in
// use; a further group costs planes of partial sums, so it has to raise that
// share by `plane_cost`.  The fewest groups always qualify, so a layout is found
// for every nz.
inline PssfpWorkgroup pssfp_workgroup(int nz, int lanes, int most, double plane_cost) {
    PssfpWorkgroup layout {0, 0, 0};
    double best = 0.0;
    const int least = (nz + most - 1) / most;
    for (int g = least; g <= least + 5 && g <= nz; g++) {
        const int zg = (nz + g - 1) / g;
        if ((nz + zg - 1) / zg != g) continue;
        const int vb = lanes / zg;
        const double share = double(vb) * nz / g / lanes - plane_cost * g;
        if (layout.groups == 0 || share > best) {
            best = share;
            layout = {vb, zg, g};
        }
    }
    return layout;
}

}  // namespace compas
