// kernels_fast_b2_c2_abs.hip -- register-resident outlier kernels, 16-bit, 2 channel(s), absolute
// thresholds.
#include "kernels_fast.h"

namespace cp {

bool launch_fast_b2_c2_abs(const OutlierK& k, int shape, hipStream_t s) { return launch_fast_c<true, 2, 2>(k, shape, s); }

}  // namespace cp
