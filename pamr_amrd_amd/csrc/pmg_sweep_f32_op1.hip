// pmg_sweep_f32_op1.hip -- the fused sweep's tile variants, float, operator 1.
#define PMG_SWEEP_IMPL
#include "pmg_sweep_launch.h"

namespace pmg {
template int launch_sweep<float, 1, false>(hipStream_t, int, SweepP<float>, bool, bool);
template int launch_sweep<float, 1, true>(hipStream_t, int, SweepP<float>, bool, bool);
}  // namespace pmg
