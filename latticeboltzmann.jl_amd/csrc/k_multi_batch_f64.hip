// k_multi_batch_f64.hip -- batched periodic D2Q9 lattices, several steps per pass, storage f64.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_BATCH_BLOCK(f64, StF64, 9)
}  // namespace lbm
