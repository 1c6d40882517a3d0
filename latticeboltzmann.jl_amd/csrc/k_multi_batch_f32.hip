// k_multi_batch_f32.hip -- batched periodic D2Q9 lattices, several steps per pass, storage f32.
// FP32 arithmetic: compiled with -ffp-contract=fast.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_BATCH_BLOCK(f32, StF32, 9)
}  // namespace lbm
