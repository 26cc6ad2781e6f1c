// kernels_fast_b2_c4_abs.hip -- register-resident outlier kernels, 16-bit, 4 channel(s), absolute
// thresholds.
#include "kernels_fast.h"

namespace cp {

bool launch_fast_b2_c4_abs(const OutlierK& k, int shape, hipStream_t s) { return launch_fast_c<true, 2, 4>(k, shape, s); }

}  // namespace cp
