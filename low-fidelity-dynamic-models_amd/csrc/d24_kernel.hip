// 24-DOF integration kernels: every tire model x control source instantiation.
#include "integrate.h"

namespace lfdm {

hipError_t launch_d24(const Launch& L, int block, hipStream_t stream) {
    if (L.S <= 0 || L.nsteps <= 0) return hipSuccess;
    if (L.lanes > 1 && !L.strict) return launch_d24_group(L, block, stream);
    return kern::launch_model<kern::M24>(L, block, stream);
}

}  // namespace lfdm
