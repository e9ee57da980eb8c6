// pmg_small_f32.hip -- the small-level legs of the V-cycle, float.
#define PMG_SMALL_IMPL
#include "pmg_small.h"

namespace pmg {
template int launch_small<float>(hipStream_t, int, SmallP<float>, int, bool, bool);
}  // namespace pmg
