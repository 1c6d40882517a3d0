// k_multi_f64_q4_5.hip -- several fused steps per pass, storage f64, D2Q{4,5}.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI(f64, StF64, 4)
LBM_DEFINE_MULTI(f64, StF64, 5)
}  // namespace lbm
