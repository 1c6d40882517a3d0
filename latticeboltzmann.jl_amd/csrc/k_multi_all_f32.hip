// k_multi_all_f32.hip -- several fused steps per pass that keep every step's field,
// periodic SRT lattices, storage f32.
#include "lbm_multi.h"

namespace lbm {
int run_multi_all_f32(const MultiLaunch &L, const LevelOut &o, const StepParams<float> &p,
                      hipStream_t s) {
    return launch_all_any<StF32>(L, o, p, s);
}
}  // namespace lbm
