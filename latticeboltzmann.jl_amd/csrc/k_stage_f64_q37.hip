// k_stage_f64_q37.hip -- several fused steps per pass, storage f64, D2Q37.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_stage.h"

namespace lbm {
LBM_DEFINE_STAGES(f64, StF64, 37)
}  // namespace lbm
