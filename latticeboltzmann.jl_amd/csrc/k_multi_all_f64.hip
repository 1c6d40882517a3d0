// k_multi_all_f64.hip -- several fused steps per pass that keep every step's field,
// periodic SRT/TRT lattices, storage f64.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI_ALL(f64, StF64)
}  // namespace lbm
