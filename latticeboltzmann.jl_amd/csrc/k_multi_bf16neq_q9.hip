// k_multi_bf16neq_q9.hip -- several fused steps per pass, storage bf16neq, D2Q9.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI(bf16neq, StBF16Neq, 9)
}  // namespace lbm
