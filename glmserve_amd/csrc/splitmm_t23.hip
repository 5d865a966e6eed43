#include "splitmm_launch.hpp"

namespace glmmoe {
template int sm_moe<23>(bool, bool, int, const SmArgs&, unsigned, hipStream_t);
template int sm_dense<23>(bool, const SmArgs&, hipStream_t);
}  // namespace glmmoe
