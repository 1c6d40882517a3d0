// k_stage_f64_q21.hip -- several fused steps per pass, storage f64, D2Q21.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_stage.h"

namespace lbm {
LBM_DEFINE_STAGES(f64, StF64, 21)
}  // namespace lbm
