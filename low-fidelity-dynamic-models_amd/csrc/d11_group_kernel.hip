// 11-DOF integration kernels on lane groups: every tire model x control source instantiation.
#include "integrate_group.h"

namespace lfdm {

hipError_t launch_d11_group(const Launch& L, int block, hipStream_t stream) {
    if (L.waves == 1) return kern::launch_tire<kern::M11g<true>, 1>(L, block, stream);
    return kern::launch_tire<kern::M11g<false>, 2>(L, block, stream);
}

}  // namespace lfdm
