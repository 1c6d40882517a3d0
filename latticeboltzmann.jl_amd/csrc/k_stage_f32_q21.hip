// k_stage_f32_q21.hip -- several fused steps per pass, storage f32, D2Q21.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_stage.h"

namespace lbm {
LBM_DEFINE_STAGES(f32, StF32, 21)
}  // namespace lbm
