// Stop flag of the COCG iterations (Scal::done).
//
// A kernel that finishes the scalars of an iteration may find that the recursion
// stops, and then stores the flag while other workgroups of the same launch have not
// read it yet.  Were any non-zero value a reason to return, the waves of one of those
// workgroups could read different values: some would leave before its barrier and the
// others would decide on partial sums that were never written.  The flag therefore
// names the launch that set it, and its own launch does not count it: there every
// workgroup comes to the same decision from the same partial sums.
#pragma once

#include <cstdint>

namespace pg {

// set outside the vector kernels (a kernel of one workgroup, the host)
constexpr int32_t kStopOther = 1;
// iteration k of a batch: the kernel that forms p, and the one that forms r and z
constexpr int32_t stop_direction(int k) { return 2 * k + 2; }
constexpr int32_t stop_update(int k) { return 2 * k + 3; }
// whether launch `self` finds the recursion stopped by an earlier one; every wave of the
// launch gets the same answer whenever it reads the flag
constexpr bool stopped_before(int32_t flag, int32_t self) { return flag != 0 && flag != self; }

}  // namespace pg
