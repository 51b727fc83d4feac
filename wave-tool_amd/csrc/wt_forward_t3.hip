// Plain forward kernel (every launch shape) and batched kernel, texture mode kTexR8Repeat.
#include "wt_forward.hpp"

namespace wt {
hipError_t launch_forward_t3(const FwdParams& p, const LaunchShape& s, hipStream_t st) {
  return launch_forward_mode<kTexR8Repeat>(p, s, st);
}
hipError_t launch_forward_batched_t3(const BatchArgs& a, hipStream_t st) {
  return launch_batched_mode<kTexR8Repeat>(a, st);
}
}  // namespace wt
