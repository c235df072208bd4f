// The complex FISP recursion with one lane per voxel (see fisp.hip).

#include "compas/device/fisp_launch.h"

namespace compas {

FispLauncher fisp_epg_launcher_1(int spl) {
    return find_fisp_epg<1, 1, 32>(spl);
}

}  // namespace compas
