// pmg_small_f64.hip -- the small-level legs of the V-cycle, double.
#define PMG_SMALL_IMPL
#include "pmg_small.h"

namespace pmg {
template int launch_small<double>(hipStream_t, int, SmallP<double>, int, bool, bool);
}  // namespace pmg
