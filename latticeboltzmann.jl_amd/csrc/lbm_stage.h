// lbm_stage.h -- several fused time steps per pass on the stencils that reach
// two or three nodes (D2Q13/17/21/37), FP64 and FP32.
//
// A single step of these sets is bound by its 2 Q sizeof(population) bytes per
// node (D2Q37 FP64 2048 x 1024: 1.24 GB a step, 4.9 TB/s).  k_stages advances T
// steps per pass: the block is a pipeline of T groups of waves on the same 128
// columns, group l computes step l + 1 of a row, M + 1 rows behind group l - 1
// (M: the stencil's reach), and hands its rows on through rings in LDS.
//
// 2048 x 1024 nodes between two walls, SRT, us a step, single steps / pipeline:
//   FP64: D2Q13 91 / 38, D2Q17 121 / 55, D2Q21 184 / 100, D2Q37 255 / 158;
//   FP32: D2Q13 46 / 29, D2Q17 61 / 39, D2Q21 90 / 49, D2Q37 130 / 65.
// D2Q37 FP64 moves 3.9 TB/s: a row and step takes 830 FP64 instructions, and the
// rings leave room for two waves per SIMD, which wait 59 % of their cycles for
// loads and at the barriers: latency bounds it, not the rate of memory.
//
// SUB = 2 (FP64): two sub-groups take a group's rows in turn, each row over two
// iterations, which doubles the waves that the same rings feed: D2Q13 42.9 -> 40.7,
// D2Q17 65 -> 59, D2Q37 172 -> 170.  FP32 has room for several blocks per CU
// instead and loses by it (D2Q37 71 -> 78).
//
// What is not waited for matters most here: the next row's loads stay in flight
// across the barriers as long as no later load is waited for, so everything else
// that a row reads from memory (force, walls) comes before them (D2Q17 FP64
// 78 -> 59 us), and a row goes straight from one of two buffers, never copied.
#pragma once

#include "lbm_multi.h"

namespace lbm {

// A population that moves up by c_y is read M + c_y rows after it was written:
// its ring holds M + c_y + 1 rows, and the reader of row k's turn takes the
// slot that the writer fills next (read, barrier, write, barrier).  D2Q37 FP64:
// 148 rows of 134 columns, 155 KB of the CU's 160.
template <int QID, class ST, int T, int SUB>
struct StageShape {
    using V = typename ST::T;
    static constexpr int Q = QT<QID>::Q, M = QT<QID>::MAXC;
    static constexpr int COLS = kStageCols;
    static constexpr int PITCH = COLS + 2 * M;  // end lanes read and write M beyond
    static constexpr int HX = M * (T - 1);
    // columns written: stores end on transaction boundaries
    static constexpr int OUT = stage_out(M, T, (int)sizeof(typename ST::store_t));
    static_assert(OUT > 0, "halo wider than the block");
    LBM_HD static constexpr int depth(int i) { return M + QT<QID>::cy(i) + 1; }
    LBM_HD static constexpr int row0(int i) {
        int n = 0;
        for (int j = 0; j < i; ++j) n += depth(j);
        return n;
    }
    static constexpr int ROWS = row0(Q);
    static constexpr int ELEMS = (T - 1) * ROWS * PITCH;
    static_assert(ELEMS * sizeof(V) <= 160 * 1024, "LDS of a CU");
    static constexpr int LAG = 2 * M + SUB;  // iterations from one group's first row to the next one's
};

struct StageArgs {
    int tiles_x, tiles, chunk;  // strips of columns x chunks of rows, dealt by XCD
    int rows;                   // rows per chunk
    int first;                  // the first step collides S_0 in place
    int north;                  // the list holds a north wall
};

// Walls (north and south ones; other lists keep single steps).  A wall
// replaces a population whose source lies beyond it by the node's own
// post-collision opposite.  North: the reader takes it from the opposite's
// ring, where the reader's own row is still kept.  South: the writer of row
// y < c_y puts it into the slot and column that the reader will pull: the slot
// of a row that wraps around.  Beyond the upper end (rows ny, ny + 1, ...) that
// would be a row whose own values a north wall still reads: there it is left
// out, and rows beyond an end hold other values than the lattice's.  Two steps
// never read them; three do, so both walls together must span the lattice,
// which replaces all that is pulled from there.
template <int QID, int COLL, class ST, int T, int SUB, bool BC>
__global__ void __launch_bounds__(kStageCols * SUB * T)
k_stages(const typename ST::store_t *__restrict__ C, typename ST::store_t *__restrict__ Cn,
         const StepParams<typename ST::T> p, const MultiConsts<typename ST::T> mc,
         const StageArgs a) {
    using V = typename ST::T;
    using S = typename ST::store_t;
    using SH = StageShape<QID, ST, T, SUB>;
    constexpr int Q = SH::Q, M = SH::M, PITCH = SH::PITCH;
    __shared__ V ring[SH::ELEMS];
    const int tile = tile_of_block(a);
    if (tile >= a.tiles) return;  // whole blocks
    const int group = __builtin_amdgcn_readfirstlane((int)threadIdx.x / SH::COLS);
    const int stage = group / SUB, part = group - stage * SUB;
    const int c = (int)threadIdx.x - group * SH::COLS;
    const int chunk = tile / a.tiles_x, strip = tile - chunk * a.tiles_x;
    const int y0 = chunk * a.rows, y1 = min(y0 + a.rows, p.ny);
    const int xo = strip * SH::OUT, col = xo - SH::HX + c;
    const int x = wrap(col, p.nx);
    const bool out = col >= xo && col < min(xo + SH::OUT, p.nx);
    // byte offsets of the columns that a pull reads: x - d at offs[M + d]
    unsigned offs[2 * M + 1];
#pragma unroll
    for (int d = -M; d <= M; ++d)
        offs[M + d] = (unsigned)(a.first ? x : wrap(x - d, p.nx)) * (unsigned)sizeof(S);
    V *const mine = ring + c + M;  // the lane's column
    // The byte offsets and the plane stride are hidden from the optimiser, which
    // would otherwise keep Q plane addresses in registers and spill them.
    auto fetch = [&](int row, S(&pre)[Q]) {
        long long rs[2 * M + 1];
        unsigned o[2 * M + 1];
#pragma unroll
        for (int d = -M; d <= M; ++d) {
            rs[M + d] = (long long)p.nx * __builtin_amdgcn_readfirstlane(a.first ? row : wrap(row - d, p.ny));
            o[M + d] = offs[M + d];
            asm volatile("" : "+v"(o[M + d]));
        }
        const long long plane = opaque_uniform(p.plane);
        const S *base = C;
        auto one = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            pre[i] = ld_g(at_b(base + rs[M + QT<QID>::cy(i)], o[M + QT<QID>::cx(i)]));
            base += plane;
        };
        adj_each_node<QID>(one);
    };
    // Rows of this group, unwrapped: v, v + SUB, ... below hi, one every SUB
    // iterations from `start` on; slot[s] = iteration mod s.  A row is pulled in
    // its first iteration and put into the rings in its last one.
    int v = y0 - M * (T - 1 - stage) + part;
    const int hi = y1 + M * (T - 1 - stage);
    int row = __builtin_amdgcn_readfirstlane(wrap(v, p.ny));
    const int start = stage * SH::LAG + part, iters = (y1 - y0) + (T - 1) * SH::LAG + SUB - 1;
    const int end = start + (hi - v + SUB - 1) / SUB * SUB;
    int slot[2 * M + 2];
#pragma unroll
    for (int s = 1; s <= 2 * M + 1; ++s) slot[s] = __builtin_amdgcn_readfirstlane(start % s);
    auto row_after = [&](int r) { return __builtin_amdgcn_readfirstlane(r + SUB >= p.ny ? r + SUB - p.ny : r + SUB); };
    auto advance = [&] {
        v += SUB;
        row = row_after(row);
    };
    auto turn = [&] {  // to the next iteration
#pragma unroll
        for (int s = 1; s <= 2 * M + 1; ++s)
            slot[s] = __builtin_amdgcn_readfirstlane(slot[s] + 1 == s ? 0 : slot[s] + 1);
    };
    // The row's force, read (as the walls' values are) before the loads of the
    // next row are issued: read after them it would wait for them all.
    V Fx = V(0), Fy = V(0);
    auto read_force = [&] {
        if (p.force_kind != 0) node_force_wait(p, x, row, Fx, Fy);
    };
    auto collide = [&](V(&f)[Q]) {
        constexpr int P1 = (2 * Q / 5) | 1, P2 = P1 + 4;
        collide_pairs<QID, COLL>(f, p, mc, [&](V &gx, V &gy) { gx = Fx; gy = Fy; },
                                 [&](auto Ic, V &ux, V &uy) {
                                     constexpr int i = decltype(Ic)::value;
                                     if constexpr (SUB == 2 && (i == P1 || i == P2)) {
                                         // what is done stays before the barrier, the rest after it
                                         auto done = [&](auto Jc) {
                                             constexpr int j = decltype(Jc)::value;
                                             if constexpr (j < i || QT<QID>::opp(j) < i) {
                                                 V &g = f[j];
                                                 asm volatile("" : "+v"(g));
                                             }
                                         };
                                         adj_each_node<QID>(done);
                                         __syncthreads();
                                         asm volatile("" : "+v"(ux), "+v"(uy));
                                         if constexpr (i == P1) turn();
                                     }
                                 },
                                 LBM_SEQ);
    };
    auto in_range = [&](const BCDev &bc) {
        return bc.kind == 1 || (x >= bc.x0 && x <= bc.x1 && row >= bc.y0 && row <= bc.y1);
    };
    // The row's populations pulled from beyond the north (D = 0) or south (D = 2)
    // wall: own(j) is the node's post-collision population j.  All of them are
    // read before any is used; one by one, the rows at a wall took 40 us a pass.
    auto walls = [&](auto Dc, V(&f)[Q], auto &&own) {
        constexpr int D = decltype(Dc)::value;
        V w[Q];
        auto read = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            if constexpr (D == 0 ? QT<QID>::cy(i) < 0 : QT<QID>::cy(i) > 0) w[i] = own(std::integral_constant<int, QT<QID>::opp(i)>{});
        };
        adj_each_node<QID>(read);
        for (int b = 0; b < p.nbc; ++b) {
            const BCDev bc = p.bcs[b];
            if (bc.dir != D) continue;
            const bool in = in_range(bc);
            V t[Q];
            auto copy = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                if constexpr (D == 0 ? QT<QID>::cy(i) < 0 : QT<QID>::cy(i) > 0) t[i] = w[i];
            };
            adj_each_node<QID>(copy);
            if (D == 0 && bc.kind == 1) {
                auto move = [&](auto Ic) {
                    constexpr int i = decltype(Ic)::value;
                    if constexpr (D == 0 ? QT<QID>::cy(i) < 0 : QT<QID>::cy(i) > 0) t[i] = w[i] + static_cast<V>(p.mw[b * Q + i]);
                };
                adj_each_node<QID>(move);
            }
            auto take = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value, cy = QT<QID>::cy(i);
                if constexpr (D == 0 ? QT<QID>::cy(i) < 0 : QT<QID>::cy(i) > 0) f[i] = in && (D == 0 ? row - cy >= p.ny : row - cy < 0) ? t[i] : f[i];
            };
            adj_each_node<QID>(take);
        }
    };
    // a row into the rings that the next group reads
    auto put = [&](const V(&f)[Q]) {
        V *const dst = mine + stage * (SH::ROWS * PITCH);
        auto one = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            dst[(SH::row0(i) + slot[SH::depth(i)]) * PITCH] = f[i];
        };
        adj_each_node<QID>(one);
        if constexpr (BC) {
            if (row < M && (v < p.ny || !a.north))
                for (int b = 0; b < p.nbc; ++b) {
                    const BCDev bc = p.bcs[b];
                    if (bc.dir != 2 || !in_range(bc)) continue;  // (moving walls are north ones)
                    auto south = [&](auto Ic) {
                        constexpr int i = decltype(Ic)::value, cy = QT<QID>::cy(i);
                        constexpr int j = QT<QID>::opp(i), D = SH::depth(i);
                        if constexpr (cy > 0) {
                            if (row - cy < 0) {
                                const int at = slot[D] - cy;  // cy rows before this one
                                dst[(SH::row0(i) + (at < 0 ? at + D : at)) * PITCH -
                                    QT<QID>::cx(i)] = f[j];
                            }
                        }
                    };
                    adj_each_node<QID>(south);
                }
        }
    };
    // Every group passes the two barriers of each iteration, working or not
    // (the branches on the group are wave-uniform).
#pragma unroll 1
    for (int k = 0; k < start; ++k) {
        __syncthreads();
        __syncthreads();
    }
    if (stage == 0) {
        // a row is loaded while the one before it collides; two buffers in turn
        S pre[2][Q];
        auto one_row = [&](S(&now)[Q], S(&then)[Q]) {
            V f[Q];
            auto dec = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                f[i] = ST::decode(now[i], i, p);
            };
            adj_each_node<QID>(dec);
            read_force();
            if constexpr (BC) {
                auto own = [&](auto Jc) {
                    constexpr int j = decltype(Jc)::value;
                    return ST::decode(ld_g(at_b(C + p.plane * j + (long long)p.nx * row, offs[M])), j, p);
                };
                if (!a.first && row >= p.ny - M) walls(std::integral_constant<int, 0>{}, f, own);
                if (!a.first && row < M) walls(std::integral_constant<int, 2>{}, f, own);
            }
            fetch(row_after(row), then);
            __syncthreads();
            collide(f);
            put(f);
            __syncthreads();
            turn();
            advance();
        };
        fetch(row, pre[0]);
#pragma unroll 1
        while (v < hi) {
            one_row(pre[0], pre[1]);
            if (v >= hi) break;
            one_row(pre[1], pre[0]);
        }
    } else {
        V *const src = mine + (stage - 1) * (SH::ROWS * PITCH);
#pragma unroll 1
        while (v < hi) {
            V f[Q];
            read_force();
            auto pull = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                f[i] = src[(SH::row0(i) + slot[SH::depth(i)]) * PITCH - QT<QID>::cx(i)];
            };
            adj_each_node<QID>(pull);
            if constexpr (BC) {
                auto own = [&](auto Jc) {
                    constexpr int j = decltype(Jc)::value, D = SH::depth(j);
                    const int at = slot[D] + QT<QID>::cy(j);  // M + 1 rows before slot[D]
                    return src[(SH::row0(j) + (at >= D ? at - D : at)) * PITCH];
                };
                if (row >= p.ny - M) walls(std::integral_constant<int, 0>{}, f, own);
            }
            __syncthreads();
            collide(f);
            if (stage == T - 1) {
                if (out) {
                    const long long plane = opaque_uniform(p.plane);
                    S *base = Cn + (long long)p.nx * row;
                    unsigned o = offs[M];
                    asm volatile("" : "+v"(o));
                    auto st = [&](auto Ic) {
                        constexpr int i = decltype(Ic)::value;
                        Pack<S, 1> pk;
                        pk.v[0] = ST::encode(f[i], i, p);
                        put_pack<true, S, 1>(at_b(base, o), pk);
                        base += plane;
                    };
                    adj_each_node<QID>(st);
                }
            } else {
                put(f);
            }
            __syncthreads();
            turn();
            advance();
        }
    }
    // the iterations after this group's last row
#pragma unroll 1
    for (int k = end; k < iters; ++k) {
        __syncthreads();
        __syncthreads();
    }
}

template <int QID, int COLL, class ST, int T, int SUB, bool BC>
int launch_stages(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    using S = typename ST::store_t;
    using SH = StageShape<QID, ST, T, SUB>;
    if (p.nx > kMultiMaxNx || p.ny < 2 * SH::M || (L.walls & (2 | 8))) return -5;
    constexpr int threads = kStageCols * SUB * T;
    static const int slots = [] {
        int per_cu = 0, dev = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, k_stages<QID, COLL, ST, T, SUB, BC>, threads, 0) != hipSuccess ||
            hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        return per_cu * cus;
    }();
    if (slots < 1) return -4;
    StageArgs a;
    a.first = L.first;
    a.north = L.walls & 1;
    a.tiles_x = (p.nx + SH::OUT - 1) / SH::OUT;
    // one resident round of blocks, at least kStageRows rows each (a chunk
    // computes (T - 1) LAG rows of run-in)
    const int down = slots / a.tiles_x > 0 ? slots / a.tiles_x : 1;
    a.rows = (p.ny + down - 1) / down;
    if (a.rows < kStageRows) a.rows = kStageRows;
    const unsigned blocks = deal_tiles(a, (p.ny + a.rows - 1) / a.rows);
    k_stages<QID, COLL, ST, T, SUB, BC><<<blocks, threads, 0, s>>>(
        static_cast<const S *>(L.src), static_cast<S *>(L.dst), p, multi_consts(p), a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <int QID, int COLL, class ST, bool BC>
int launch_stages_t(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    constexpr bool f64 = sizeof(typename ST::T) == 8;
    constexpr int most = stage_steps(QID, f64), SUB = f64 ? 2 : 1;
    if (L.kernel != kMultiStages) return -5;
    if (L.steps == 2) return launch_stages<QID, COLL, ST, 2, SUB, BC>(L, p, s);
    if constexpr (most >= 3)
        if (L.steps == 3) return launch_stages<QID, COLL, ST, 3, SUB, BC>(L, p, s);
    return -5;
}

template <int QID, class ST>
int launch_stages_any(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    const bool bc = p.nbc > 0;
    switch (L.coll) {
    case 0: return bc ? launch_stages_t<QID, 0, ST, true>(L, p, s) : launch_stages_t<QID, 0, ST, false>(L, p, s);
    case 1: return bc ? launch_stages_t<QID, 1, ST, true>(L, p, s) : launch_stages_t<QID, 1, ST, false>(L, p, s);
    default: return -2;
    }
}

#define LBM_DEFINE_STAGES(TAG, ST, QID)                                                     \
    int run_multi_##TAG##_q##QID(const MultiLaunch &L, const StepParams<typename ST::T> &p, \
                                 hipStream_t s) {                                           \
        return launch_stages_any<QID, ST>(L, p, s);                                         \
    }

}  // namespace lbm
