// k_stage_f32_q17.hip -- several fused steps per pass, storage f32, D2Q17.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_stage.h"

namespace lbm {
LBM_DEFINE_STAGES(f32, StF32, 17)
}  // namespace lbm
