// m27q_wide_q80.hip -- the instances of m27q_wide.h for one weight type (one
// file per type, so that they compile in parallel).
#include "m27q_wide.h"

namespace m27q {

hipError_t launch_wide_q80(int layout, const MatmulMultiParams &p, hipStream_t s) { return launch_wide_l<WQ80>(layout, p, s); }

}  // namespace m27q
