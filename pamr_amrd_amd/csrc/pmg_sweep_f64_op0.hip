// pmg_sweep_f64_op0.hip -- the fused sweep's tile variants, double, operator 0.
#define PMG_SWEEP_IMPL
#include "pmg_sweep_launch.h"

namespace pmg {
template int launch_sweep<double, 0, false>(hipStream_t, int, SweepP<double>, bool, bool);
template int launch_sweep<double, 0, true>(hipStream_t, int, SweepP<double>, bool, bool);
}  // namespace pmg
