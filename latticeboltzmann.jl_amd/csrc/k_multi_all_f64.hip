// k_multi_all_f64.hip -- several fused steps per pass that keep every step's field,
// periodic SRT/TRT lattices, storage f64.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_multi.h"

namespace lbm {
int run_multi_all_f64(const MultiLaunch &L, const LevelOut &o, const StepParams<double> &p,
                      hipStream_t s) {
    return launch_all_any<StF64>(L, o, p, s);
}
}  // namespace lbm
