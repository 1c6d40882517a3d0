// k_multi_all_f32.hip -- several fused steps per pass that keep every step's field,
// periodic SRT/TRT lattices, storage f32.
#include "lbm_multi.h"

namespace lbm {
LBM_DEFINE_MULTI_ALL(f32, StF32)
}  // namespace lbm
