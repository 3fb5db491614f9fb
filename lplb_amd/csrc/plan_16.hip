// One-launch plans of groups of up to 16 ranks (see plan_kernel.h).
#include "plan_kernel.h"

namespace lplb {

int launch_plan_up_to_16(PlanArgs &a, hipStream_t s, bool *done) {
  if (a.sh.D <= 1)
    return launch_plan_padded_or_not<16, 1>(a, s, done);
  if (a.sh.D <= 2)
    return launch_plan_padded_or_not<16, 2>(a, s, done);
  return LPLB_OK;
}

int scan_and_solve_up_to_16(const ScanSolveArgs &a, hipStream_t s) {
  return a.solve.D <= 1 ? launch_scan_and_solve<16, 1>(a, s) : launch_scan_and_solve<16, 2>(a, s);
}

} // namespace lplb
