#include "splitmm_launch.hpp"

namespace glmmoe {
template int sm_moe<13>(bool, bool, int, const SmArgs&, unsigned, hipStream_t);
template int sm_dense<13>(bool, const SmArgs&, hipStream_t);
}  // namespace glmmoe
