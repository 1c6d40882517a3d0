// k_multi_mei_f64.hip -- steps of the iterative initialization (collide with the
// prescribed velocity, stream, boundary list, density check), storage f64.
// Plain FP64: compiled with -ffp-contract=off (bit-exact with the CPU restatement).
#include "lbm_multi.h"

namespace lbm {

// One step C_(t-1) -> C_t with the check of S_t.  Small lattices are bound by
// the launch; what counts is that a step is one launch and no host round trip:
// collide, stream, gather and a wait for the copy took 29 us a step on 128 x 128
// D2Q9 nodes, whatever the size.
template <int QID>
__global__ void __launch_bounds__(256)
k_mei_step(const double *__restrict__ C, double *__restrict__ Cn, const StepParams<double> p,
           const MeiStop stop) {
    if (mei_done(stop)) return;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= p.nx) return;
    double f[QT<QID>::Q];
    pull_seq<QID, StF64>(C, p, x, y, f, LBM_SEQ);
    if (x == p.nx - 1 && y == p.ny - 1) mei_check<QID>(stop, f, stop.step);
    collide_mei_node<QID>(f, p, x, y);
    store_local<QID, StF64>(Cn, p, (long long)x + (long long)p.nx * y, f, LBM_SEQ);
}

template <int QID>
static int mei_step(const double *src, double *dst, const StepParams<double> &p,
                    const MeiStop &stop, hipStream_t s) {
    const int block = p.nx >= 256 ? 256 : (p.nx > 64 ? 128 : 64);
    const dim3 grid((unsigned)((p.nx + block - 1) / block), (unsigned)p.ny);
    k_mei_step<QID><<<grid, block, 0, s>>>(src, dst, p, stop);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int run_mei_step(int qid, const double *src, double *dst, const StepParams<double> &p,
                 const MeiStop &stop, hipStream_t s) {
    switch (qid) {
    case 4: return mei_step<4>(src, dst, p, stop, s);
    case 5: return mei_step<5>(src, dst, p, stop, s);
    case 9: return mei_step<9>(src, dst, p, stop, s);
    case 13: return mei_step<13>(src, dst, p, stop, s);
    case 17: return mei_step<17>(src, dst, p, stop, s);
    case 21: return mei_step<21>(src, dst, p, stop, s);
    case 37: return mei_step<37>(src, dst, p, stop, s);
    default: return -1;
    }
}

int run_mei_tile(const MultiLaunch &L, const StepParams<double> &p, hipStream_t s) {
    switch (L.qid * 2 + (L.walls != 0)) {
    case 8: return launch_tile<4, 3, StF64, false>(L, p, s);
    case 9: return launch_tile<4, 3, StF64, true>(L, p, s);
    case 10: return launch_tile<5, 3, StF64, false>(L, p, s);
    case 11: return launch_tile<5, 3, StF64, true>(L, p, s);
    case 18: return launch_tile<9, 3, StF64, false>(L, p, s);
    case 19: return launch_tile<9, 3, StF64, true>(L, p, s);
    default: return -1;
    }
}

}  // namespace lbm
