// k_multi_f32_q9.hip -- several fused steps per pass, storage f32, D2Q9.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI(f32, StF32, 9)
}  // namespace lbm
