#include "splitmm_launch.hpp"

namespace glmmoe {
template int sm_moe<14>(bool, bool, int, const SmArgs&, unsigned, hipStream_t);
template int sm_dense<14>(bool, const SmArgs&, hipStream_t);
}  // namespace glmmoe
