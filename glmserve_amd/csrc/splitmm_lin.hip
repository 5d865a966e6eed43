#include "splitmm_launch.hpp"

namespace glmmoe {
template int sm_dense<kSmW4>(bool, const SmArgs&, hipStream_t);
template int sm_dense<kSmFp8>(bool, const SmArgs&, hipStream_t);
}  // namespace glmmoe
