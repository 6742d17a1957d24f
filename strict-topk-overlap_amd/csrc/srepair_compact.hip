// The one-launch repair over compact predictions (kernel and comments in
// srepair_kernel.hpp).
#include "srepair_kernel.hpp"

namespace stk {

int launch_srepair_compact(int dtype, const SRepairArgs& a, hipStream_t st) {
  return srepair_launch<true>(dtype, a, st);
}

}  // namespace stk
