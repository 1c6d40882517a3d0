// k_stage_f32_q13.hip -- several fused steps per pass, storage f32, D2Q13.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_stage.h"

namespace lbm {
LBM_DEFINE_STAGES(f32, StF32, 13)
}  // namespace lbm
