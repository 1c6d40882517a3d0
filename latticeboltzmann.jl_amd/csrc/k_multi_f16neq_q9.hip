// k_multi_f16neq_q9.hip -- several fused steps per pass, storage f16neq, D2Q9.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI(f16neq, StF16Neq, 9)
}  // namespace lbm
