// k_multi_f32_q4_5.hip -- several fused steps per pass, storage f32, D2Q{4,5}.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI(f32, StF32, 4)
LBM_DEFINE_MULTI(f32, StF32, 5)
}  // namespace lbm
