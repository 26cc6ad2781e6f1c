// kernels_fast_b2_c2_rel.hip -- register-resident outlier kernels, 16-bit, 2 channel(s), relative
// thresholds.
#include "kernels_fast.h"

namespace cp {

bool launch_fast_b2_c2_rel(const OutlierK& k, int shape, hipStream_t s) { return launch_fast_c<false, 2, 2>(k, shape, s); }

}  // namespace cp
