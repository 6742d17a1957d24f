// The one-launch repair over saved and hybrid predictions (kernel and comments
// in srepair_kernel.hpp), and the launch dispatch.
#include "srepair_kernel.hpp"

namespace stk {

bool srepair_covers(int dtype, int b, int d, int sa, int sp, int sc, uintptr_t align) {
  if (dtype != DT_BF16 && dtype != DT_F16) return false;
  if (!tok_nch(dtype, d, b, align)) return false;
  if (sa < 1 || sp < 1 || sc < 1 || sa > kTailMaxK || sp > kTailMaxK || sc > kTailMaxK)
    return false;
  const int per_pass = kTailThreads * 4 / d;
  return (sc + per_pass - 1) / per_pass <= 16;
}

int launch_srepair(int dtype, const SRepairArgs& a, hipStream_t st) {
  return a.rids ? launch_srepair_compact(dtype, a, st) : srepair_launch<false>(dtype, a, st);
}

}  // namespace stk
