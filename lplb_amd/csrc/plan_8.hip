// One-launch plans of groups of up to 8 ranks (see plan_kernel.h).
#include "plan_kernel.h"

namespace lplb {

int launch_plan_up_to_8(PlanArgs &a, hipStream_t s, bool *done) {
  if (a.sh.D <= 1)
    return launch_plan_padded_or_not<8, 1>(a, s, done);
  if (a.sh.D <= 2)
    return launch_plan_padded_or_not<8, 2>(a, s, done);
  if (a.sh.D <= 4)
    return launch_plan_padded_or_not<8, 4>(a, s, done);
  return LPLB_OK;
}

int scan_and_solve_up_to_8(const ScanSolveArgs &a, hipStream_t s) {
  return a.solve.D <= 1 ? launch_scan_and_solve<8, 1>(a, s) : a.solve.D <= 2 ? launch_scan_and_solve<8, 2>(a, s) : launch_scan_and_solve<8, 4>(a, s);
}

} // namespace lplb
