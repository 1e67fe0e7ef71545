// The kernel of oxq_gemm_direct.hpp on three and four token tiles a work group.
#include "oxq_gemm_direct_launch.hpp"

namespace oxq {

hipError_t launch_direct_wide(uint32_t type, uint32_t tt, const GemmArgs &a, hipStream_t stream) {
    return launch_direct_of<3, 4>(type, tt, a, stream);
}

}  // namespace oxq
