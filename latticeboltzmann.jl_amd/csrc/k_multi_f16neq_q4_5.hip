// k_multi_f16neq_q4_5.hip -- several fused steps per pass, storage f16neq, D2Q{4,5}.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI(f16neq, StF16Neq, 4)
LBM_DEFINE_MULTI(f16neq, StF16Neq, 5)
}  // namespace lbm
