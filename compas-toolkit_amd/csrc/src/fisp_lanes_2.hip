// The complex FISP recursion with two lanes per voxel (see fisp.hip).

#include "compas/device/fisp_launch.h"

namespace compas {

FispLauncher fisp_epg_launcher_2(int spl) {
    return find_fisp_epg<2, 1, 32>(spl);
}

}  // namespace compas
