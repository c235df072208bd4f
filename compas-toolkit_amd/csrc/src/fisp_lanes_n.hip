// The complex FISP recursion with four and eight lanes per voxel (see fisp.hip).

#include "compas/device/fisp_launch.h"

namespace compas {

FispLauncher fisp_epg_launcher_n(int lpv, int spl) {
    switch (lpv) {
        case 4: return find_fisp_epg<4, 1, 16>(spl);
        case 8: return find_fisp_epg<8, 2, 16>(spl);
        default: return nullptr;
    }
}

}  // namespace compas
