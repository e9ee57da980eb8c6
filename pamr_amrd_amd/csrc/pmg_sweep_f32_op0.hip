// pmg_sweep_f32_op0.hip -- the fused sweep's tile variants, float, operator 0.
#define PMG_SWEEP_IMPL
#include "pmg_sweep_launch.h"

namespace pmg {
template int launch_sweep<float, 0, false>(hipStream_t, int, SweepP<float>, bool, bool);
template int launch_sweep<float, 0, true>(hipStream_t, int, SweepP<float>, bool, bool);
}  // namespace pmg
