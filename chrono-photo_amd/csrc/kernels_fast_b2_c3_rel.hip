// kernels_fast_b2_c3_rel.hip -- register-resident outlier kernels, 16-bit, 3 channel(s), relative
// thresholds.
#include "kernels_fast.h"

namespace cp {

bool launch_fast_b2_c3_rel(const OutlierK& k, int shape, hipStream_t s) { return launch_fast_c<false, 2, 3>(k, shape, s); }

}  // namespace cp
