// k_stage_f64_q17.hip -- several fused steps per pass, storage f64, D2Q17.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_stage.h"

namespace lbm {
LBM_DEFINE_STAGES(f64, StF64, 17)
}  // namespace lbm
