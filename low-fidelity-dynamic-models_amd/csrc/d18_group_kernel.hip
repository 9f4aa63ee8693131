// 18-DOF integration kernels on lane groups: every tire model x control source instantiation.
#include "integrate_group.h"

namespace lfdm {

hipError_t launch_d18_group(const Launch& L, int block, hipStream_t stream) {
    if (L.lanes == 4) {
        if (L.waves == 1) return kern::launch_tire<kern::M18g<4, true>, 1>(L, block, stream);
        return kern::launch_tire<kern::M18g<4, false>, 2>(L, block, stream);
    }
    return kern::launch_tire<kern::M18g<2, false>, 2>(L, block, stream);
}

}  // namespace lfdm
