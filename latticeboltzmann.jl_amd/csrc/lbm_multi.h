// lbm_multi.h -- several fused time steps per launch (temporal blocking).
//
// One fused step moves every population through HBM once; a run of n steps is
// bound by 2 Q sizeof(population) n bytes per node.  The kernels here advance
// a region by T steps per pass instead, recomputing a halo that shrinks by
// the stencil's reach per step, so T steps cost one pass:
//   * k_tile: a block keeps a tile of the lattice in LDS (small lattices);
//   * k_block: a block of waves keeps 64 columns of rows in registers and
//     exchanges the waves' edge rows through LDS (those in between);
//   * k_march: a wave marches up a strip of columns with the rows of the T
//     levels in registers and in its own LDS (large ones).
// Every node is updated by the operations of the single-step kernels in their
// order, wrapped to its lattice position, boundary list included: FP64 results
// are bit-identical to running the steps one by one.
#pragma once

#include "lbm_kernels.h"

namespace lbm {

// Constants of the pair-form collision: halves of s^2, -s and of the TRT rates
// (scaling by a power of two is exact, so folding the 1/2 of the reference's
// expressions into them changes no rounding), and -2 w per population for the
// FP32 form.
template <class T>
struct MultiConsts {
    T hs2, hns, homs, homa;
    T w2[37];
};

template <class T>
inline MultiConsts<T> multi_consts(const StepParams<T> &p) {
    MultiConsts<T> m;
    m.hs2 = T(0.5) * p.s2;
    m.hns = T(0.5) * p.neg_s;
    m.homs = T(0.5) * p.oms;
    m.homa = T(0.5) * p.oma;
    for (int i = 0; i < 37; ++i) m.w2[i] = T(-2) * p.w[i];
    return m;
}

// first population with the same weight (the same |c| components)
template <int QID>
LBM_HD constexpr int weight_rep(int i) {
    const auto ab = [](int v) { return v < 0 ? -v : v; };
    const int a = ab(QT<QID>::cx(i)), b = ab(QT<QID>::cy(i));
    for (int j = 0; j < i; ++j) {
        const int c = ab(QT<QID>::cx(j)), d = ab(QT<QID>::cy(j));
        if ((a == c && b == d) || (a == d && b == c)) return j;
    }
    return i;
}

// mx / r and my / r, correctly rounded: one refined reciprocal for both
// quotients, each finished with the exact remainder of its product (the
// division expansion's own steps, with the reciprocal shared).  Outside
// 2^-510 < r < 2^510 the plain divisions run.  A numerator small enough for
// its remainder to underflow (|m| < 2^-960) gives a velocity whose products
// vanish against 1 in the equilibrium, so its last bit never reaches a
// population.
__device__ __forceinline__ void div2(double mx, double my, double r, double &ux, double &uy) {
    double y = __builtin_amdgcn_rcp(r);
    y = __builtin_fma(y, __builtin_fma(-r, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-r, y, 1.0), y);
    const double qx = mx * y, qy = my * y;
    ux = __builtin_fma(__builtin_fma(-r, qx, mx), y, qx);
    uy = __builtin_fma(__builtin_fma(-r, qy, my), y, qy);
    const unsigned hi = static_cast<unsigned>(__double2hiint(r));
    if (__builtin_expect(hi - 0x20100000u >= 0x3fc00000u, 0)) {
        ux = mx / r;
        uy = my / r;
    }
}

// node_force, a field's values waited for in the branch that loads them: waited
// for where the branches meet, a run without a field would wait there too, for
// all its loads and stores in flight (D2Q9 FP64 4096^2: 135 -> 130 us a step).
template <class T>
__device__ __forceinline__ void node_force_wait(const StepParams<T> &p, int x, int y, T &Fx, T &Fy) {
    if (p.force_kind == 1) {
        Fx = p.Fx;
        Fy = p.Fy;
    } else {
        node_force(p, x, y, Fx, Fy);
        asm volatile("" : "+v"(Fx), "+v"(Fy));
    }
}

// node_moments with the shared reciprocal
template <int QID, int... Is>
__device__ __forceinline__ void moments_div2(const double (&f)[QT<QID>::Q], double &rho, double &ux,
                                             double &uy, std::integer_sequence<int, Is...>) {
    double mx = 0.0, my = 0.0;
    rho = f[0] + f[1];
    ((rho = (Is >= 2 ? rho + f[Is] : rho)), ...);
    ((mx = (QT<QID>::cx(Is) != 0 ? mx + cmul<QT<QID>::cx(Is)>(f[Is]) : mx)), ...);
    ((my = (QT<QID>::cy(Is) != 0 ? my + cmul<QT<QID>::cy(Is)>(f[Is]) : my)), ...);
    div2(mx, my, rho, ux, uy);
}

// collide! of one node, one opposite pair (i, j) at a time: c_j = -c_i, so u.c,
// its powers, the terms of the expansion (the odd ones change sign) and (TRT)
// the symmetric and antisymmetric parts of the pair are formed once.  `before(i, ..)`
// runs ahead of population i's part and may touch the velocity that the rest
// depends on.  Rounding for rounding the values are those of
// collide_seq (negation and scaling by 1/2 are exact, short of overflow: a run
// whose populations pass 2^1021 may reach infinity at another step); D2Q9 TRT
// FP64 takes 137 arithmetic instructions instead of 224.
template <int QID, int COLL, class F, class H, int... Is>
__device__ __forceinline__ void collide_pairs(double (&f)[QT<QID>::Q], const StepParams<double> &p,
                                              const MultiConsts<double> &mc, F &&force, H &&before,
                                              std::integer_sequence<int, Is...>) {
    constexpr int FEQ = QT<QID>::FEQ;
    static_assert(COLL <= 1, "pair form: SRT and TRT");
    double rho, ux, uy;
    moments_div2<QID>(f, rho, ux, uy, LBM_SEQ);
    if (p.force_kind != 0) {
        double Fx, Fy;
        force(Fx, Fy);
        ux = ux + p.tau_force * Fx;  // srt.jl:54 / trt.jl:79
        uy = uy + p.tau_force * Fy;
    }
    const double usq = ux * ux + uy * uy;
    const double hq = mc.hns * usq;
    // orders three and four: the factors are those of a3 / 6 and a4 / 24 with
    // the 1/2 of s^2 (u.c)^2 / 2 carried into them
    const double q3 = 0.5 * (p.three_s * usq), q4 = p.six_s3 * usq, k4 = p.three_s2 * (usq * usq);
    double rw[QT<QID>::Q];
    auto one = [&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        constexpr int j = QT<QID>::opp(i), wr = weight_rep<QID>(i);
        before(Ic, ux, uy);
        if constexpr (wr == i) rw[i] = rho * p.w[i];
        if constexpr (i <= j) {
            const double ud = udot<QID, i>(ux, uy);
            double qi, qj;
            if constexpr (i == j) {
                double a0 = FEQ >= 2 ? 1.0 + hq : 1.0;
                if constexpr (FEQ >= 4) a0 = a0 + (1.0 / 24.0) * k4;
                qi = FEQ >= 2 ? rw[wr] * a0 : rw[wr];
                qj = qi;
            } else {
                const double a1 = p.s * ud;
                double ai = 1.0 + a1, aj = 1.0 - a1;
                if constexpr (FEQ >= 2) {
                    const double ud2 = ud * ud, m2 = mc.hs2 * ud2, h2 = m2 + hq;
                    ai = ai + h2;
                    aj = aj + h2;
                    if constexpr (FEQ >= 3) {
                        const double t3 = (2.0 * (1.0 / 6.0)) * (a1 * (m2 - q3));
                        ai = ai + t3;
                        aj = aj - t3;
                    }
                    if constexpr (FEQ >= 4) {
                        const double t4 = (1.0 / 24.0) * ((p.s4 * pow4(ud) - q4 * ud2) + k4);
                        ai = ai + t4;
                        aj = aj + t4;
                    }
                }
                qi = rw[wr] * ai;
                qj = rw[wr] * aj;
            }
            if constexpr (COLL == 0) {
                f[i] = p.omo * f[i] + p.om * qi;  // srt.jl:57-59
                if constexpr (j != i) f[j] = p.omo * f[j] + p.om * qj;
            } else if constexpr (i == j) {
                f[i] = f[i] + (-p.oms) * (f[i] - qi);
            } else {  // trt.jl:82-94
                const double gi = f[i], gj = f[j];
                const double A = (-mc.homs) * ((gi + gj) - (qi + qj));
                const double B = mc.homa * ((gi - gj) - (qi - qj));
                f[i] = gi + (A - B);
                f[j] = gj + (A + B);
            }
        }
    };
    (one(std::integral_constant<int, Is>{}), ...);
}

// The same for the FP32 storages, on shifted populations g = f - w rho0.  The
// moments are summed from the pairs' sums and differences, which the TRT
// relaxation uses again; with the even and odd parts of the pair's
// equilibrium (ev, od as in collide_neq_pairs), ns = (g_i + g_j) - 2 w ev and
// na = (g_i - g_j) - 2 w od are the relaxed parts: g_i - ns / (2 tau_s) -
// na / (2 tau_a).  D2Q9 TRT: 71 arithmetic instructions per node instead of 102,
// SRT 76 instead of 89 (form 7 and 6, see multi_form).
template <int QID, int COLL, class F, class H, int... Is>
__device__ __forceinline__ void collide_pairs(float (&f)[QT<QID>::Q], const StepParams<float> &p,
                                              const MultiConsts<float> &mc, F &&force, H &&before,
                                              std::integer_sequence<int, Is...>) {
    constexpr int FEQ = QT<QID>::FEQ, Q = QT<QID>::Q;
    static_assert(COLL <= 1 || COLL == 6 || COLL == 7, "pair form: SRT and TRT");
    float s[Q], d[Q];  // pair sums and differences, at the smaller index
    auto sums = [&](auto Ic) {
        constexpr int i = decltype(Ic)::value, j = QT<QID>::opp(i);
        if constexpr (i < j) {
            s[i] = f[i] + f[j];
            d[i] = f[i] - f[j];
        } else if constexpr (i == j) {
            s[i] = f[i];
        }
    };
    (sums(std::integral_constant<int, Is>{}), ...);
    float drho = 0.0f, mx = 0.0f, my = 0.0f;
    auto mom = [&](auto Ic) {
        constexpr int i = decltype(Ic)::value, j = QT<QID>::opp(i);
        constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
        if constexpr (i <= j) drho = drho + s[i];
        if constexpr (i < j && cx != 0) mx = mx + cmul<cx>(d[i]);
        if constexpr (i < j && cy != 0) my = my + cmul<cy>(d[i]);
    };
    (mom(std::integral_constant<int, Is>{}), ...);
    const float rho = p.rho0 + drho, ir = rcp_fast(rho);
    float ux = mx * ir, uy = my * ir;
    if (p.force_kind != 0) {
        float Fx, Fy;
        force(Fx, Fy);
        ux = ux + p.tau_force * Fx;
        uy = uy + p.tau_force * Fy;
    }
    // the record form of the equilibrium (make_rec); orders three and four: the
    // even and odd powers of node_eq's polynomial in t = c.u
    float ax = ux, ay = uy, a0, a3 = 0.0f;
    NodeEq e;
    if constexpr (FEQ <= 2) {
        const float sr = p.s * rho;
        ax = sr * ux;
        ay = sr * uy;
        a0 = FEQ == 2 ? drho - 0.5f * (ax * ux + ay * uy) : drho;
        a3 = 0.5f * ir;
    } else {
        e = node_eq<QID>(drho, ux, uy, p);
        a0 = e.k0;
    }
    auto one = [&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        constexpr int j = QT<QID>::opp(i), wr = weight_rep<QID>(i);
        before(Ic, ax, ay);
        if constexpr (i == j) {
            const float n = f[i] - p.w[wr] * a0;
            if constexpr (COLL == 6) f[i] = p.omo * f[i] + p.om * (p.w[wr] * a0);
            else f[i] = f[i] - (COLL == 0 ? p.om : p.oms) * n;
        } else if constexpr (i < j) {
            float od = udot<QID, i>(ax, ay), ev = a0;
            if constexpr (FEQ == 2) {
                ev = a0 + a3 * (od * od);
            } else if constexpr (FEQ > 2) {
                const float t = od, t2 = t * t;
                od = t * (e.k1 + t2 * e.k3);
                ev = FEQ == 3 ? a0 + t2 * e.k2 : a0 + t2 * (e.k2 + t2 * e.k4);
            }
            if constexpr (COLL == 6) {  // the single-step kernels' relaxation (srt.jl:57-59)
                const float w = p.w[wr];
                f[i] = p.omo * f[i] + p.om * (w * (ev + od));
                f[j] = p.omo * f[j] + p.om * (w * (ev - od));
            } else if constexpr (COLL == 0) {
                const float w = p.w[wr];
                f[i] = f[i] - p.om * (f[i] - w * (ev + od));
                f[j] = f[j] - p.om * (f[j] - w * (ev - od));
            } else {
                const float ns = s[i] + mc.w2[wr] * ev, na = d[i] + mc.w2[wr] * od;
                if constexpr (COLL == 7) {  // one rounding at f's size instead of two
                    const float t = mc.homa * na;
                    f[i] = f[i] - (mc.homs * ns + t);
                    f[j] = f[j] - (mc.homs * ns - t);
                } else {
                    f[i] = (f[i] - mc.homs * ns) - mc.homa * na;
                    f[j] = (f[j] - mc.homs * ns) + mc.homa * na;
                }
            }
        }
    };
    (one(std::integral_constant<int, Is>{}), ...);
}

// The form of a collision (COLL 0 SRT, 1 TRT, 2 MRT; 4 SRT in the single-step
// kernels' own form): 4 and 5 that form, 6 and 7 pair forms of FP32.
//
// FP32 momentum drifts by the rounding of the weights, s sum w c^2 = 1 + d, and,
// with SRT as omo f + om feq, by that of omo = 1 - 1/tau and om: two errors that
// cancel at some tau and add up at others.  The pair form as f - om (f - feq) has
// the first only: over tau in 0.6 .. 1.0 and 200 steps its error against 64 bits
// was 0.3 to 6.4 times the single-step kernels' on D2Q9 (geometric mean 1.07), up
// to 8.6 on D2Q5 (1.9).  So SRT relaxes as they do (D2Q9 60 steps on 1500 x 1300
// 530 -> 603 us, single steps 1,754).  TRT on D2Q9 takes both relaxed parts off
// at once (at tau 0.6, where the drifts cancel, 1.05 before), on D2Q4/5, up to 1.8
// before, it runs the single-step form (5 %).  The ratio is 1.00 with each.  The
// 16-bit storages, whose single steps relax f - feq, keep the plain pairs (0.6
// to 1.02 of the single-step kernels' error) but for TRT on D2Q4/5 (up to 1.5
// before, 0.6 to 1.01).
template <int QID, int COLL, class ST>
LBM_HD constexpr int multi_form() {
    if (COLL > 1 || !ST::kShift) return COLL;
    if (COLL == 1 && QID < 9) return 5;
    return ST::kNeq ? COLL : (COLL == 0 ? 6 : 7);
}

template <int QID, int COLL, class ST, class T>
__device__ __forceinline__ void collide_multi(T (&f)[QT<QID>::Q], const StepParams<T> &p,
                                              const MultiConsts<T> &mc, int x, int y) {
    constexpr int FORM = multi_form<QID, COLL, ST>();
    if constexpr (FORM == 4 || FORM == 5) {
        collide_any<QID, FORM - 4>(f, p, x, y);
    } else if constexpr (FORM != 2) {
        collide_pairs<QID, FORM>(f, p, mc, [&](T &Fx, T &Fy) { node_force_wait(p, x, y, Fx, Fy); },
                                 [](auto, T &, T &) {}, LBM_SEQ);
    } else {
        double rho, ux, uy;
        moments_div2<QID>(f, rho, ux, uy, LBM_SEQ);
        collide_mrt_moments<QID, T>(f, p, x, y, rho, ux, uy);
    }
}

// The stop of the iterative initialization (DensityConvergence at node
// (nx, ny)), taken on the device: the thread that holds the corner compares the
// density of each new state with the previous one's and records the first step
// that converged; launches after that return at once, so the state before it
// is still in its buffer.  The output of the recording launch is not used once
// the record is set.
template <int QID, int... Is>
__device__ __forceinline__ double mei_density(const double (&f)[QT<QID>::Q],
                                              std::integer_sequence<int, Is...>) {
    double r = f[0] + f[1];
    ((Is > 1 ? (void)(r = r + f[Is]) : (void)0), ...);
    return r;
}
__device__ __forceinline__ long long mei_stopped(const MeiWatch *w) {
    return __hip_atomic_load(&w->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Whether an earlier launch recorded the stop: a launch records steps from its
// own first one up, so every thread of a launch gets the same answer, whenever
// its corner's thread records (k_tile has barriers after this).
__device__ __forceinline__ bool mei_done(const MeiStop &m) {
    const long long stop = mei_stopped(m.watch);
    return stop != 0 && stop < m.step;
}
template <int QID>
__device__ __forceinline__ void mei_check(const MeiStop &m, const double (&f)[QT<QID>::Q], long long step) {
    const double rho = mei_density<QID>(f, LBM_SEQ), d = fabs(rho - m.watch->rho);
    if (mei_stopped(m.watch) != 0) return;
    m.watch->rho = rho;
    if (d < m.eps || d > 100.0)
        __hip_atomic_store(&m.watch->stop, step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The boundary list of a node (apply_bc_seq's semantics) as a mask, formed once
// per node and pass: bit i is set when population i is replaced by the node's
// own post-collision opp(i), bit 16 + i when the last condition that replaces
// it is a moving wall (its term is added).  One-speed stencils: a wall
// replaces the populations whose component points away from it, at the row or
// column next to it.  Walking the list costs tens of dependent scalar loads
// and branches, applying the mask about 30 vector instructions: with the list
// walked at every level a 257^2 cavity ran 4.3 us per step instead of 3.3.
template <int QID>
LBM_HD constexpr unsigned wall_mask(int dir) {
    unsigned m = 0;
    for (int i = 0; i < QT<QID>::Q; ++i) {
        const int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
        if (dir == 0 ? cy < 0 : (dir == 2 ? cy > 0 : (dir == 1 ? cx < 0 : cx > 0))) m |= 1u << i;
    }
    return m;
}

// the walls of the list (bit = direction) and its last moving wall
struct WallArgs {
    int walls, moving;
};

// whether node (x, y) lies at a wall of the list
template <class T>
__device__ __forceinline__ bool at_wall(const StepParams<T> &p, int walls, int x, int y) {
    return ((walls & 1) && y == p.ny - 1) || ((walls & 2) && x == p.nx - 1) ||
           ((walls & 4) && y == 0) || ((walls & 8) && x == 0);
}

template <int QID, class T>
__device__ __forceinline__ unsigned bc_mask(const StepParams<T> &p, const BCDev *bcs, int walls, int x,
                                            int y) {
    static_assert(QT<QID>::MAXC == 1 && QT<QID>::Q <= 16, "one-speed stencils");
    unsigned m = 0;
    if (at_wall(p, walls, x, y)) {
        for (int b = 0; b < p.nbc; ++b) {
            const BCDev bc = bcs[b];
            const bool at = bc.dir == 0   ? y == p.ny - 1
                            : bc.dir == 1 ? x == p.nx - 1
                            : bc.dir == 2 ? y == 0
                                          : x == 0;
            const unsigned w = bc.dir == 0   ? wall_mask<QID>(0)
                               : bc.dir == 1 ? wall_mask<QID>(1)
                               : bc.dir == 2 ? wall_mask<QID>(2)
                                             : wall_mask<QID>(3);
            const bool inr = bc.kind == 1 || (x >= bc.x0 && x <= bc.x1 && y >= bc.y0 && y <= bc.y1);
            if (at && inr) m = (m & ~(w << 16)) | w | (bc.kind == 1 ? w << 16 : 0u);
        }
    }
    return m;
}

template <int QID, class T, class F>
__device__ __forceinline__ void bc_apply(const StepParams<T> &p, int moving, unsigned m,
                                         T (&f)[QT<QID>::Q], F &&own) {
    if (m == 0) return;
    auto one = [&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i), j = QT<QID>::opp(i);
        if constexpr (cx != 0 || cy != 0) {
            T v = own(std::integral_constant<int, j>{});
            if constexpr (cy < 0) {
                if (m & (1u << (16 + i))) v = v + static_cast<T>(p.mw[moving * QT<QID>::Q + i]);
            }
            f[i] = (m & (1u << i)) ? v : f[i];
        }
    };
    adj_each_node<QID>(one);
}

// ---------------------------------------------------------------------------
// Tiles and blocks are dealt to the 8 XCDs (workgroups go to them in turn) in
// contiguous chunks: neighbours, which read each other's halo, share an L2.
// D2Q9 TRT, us a step dealt in turn / in chunks, FP64 and FP32: tiles 160^2
// 1.92 / 1.66, 1.10 / 0.95; 64 x 16 blocks 257^2 2.55 / 1.99, 1.54 / 1.17;
// 64 x 32 blocks 512^2 4.01 / 3.61, 2.29 / 1.88; the wide ones 1021 x 517
// 7.50 / 7.11, 3.73 / 3.20.
template <class A>
__device__ __forceinline__ int tile_of_block(const A &a) {
    return (int)(blockIdx.x & 7) * a.chunk + (int)(blockIdx.x >> 3);
}
template <class A>
unsigned deal_tiles(A &a, int tiles_y) {
    a.tiles = a.tiles_x * tiles_y;
    a.chunk = (a.tiles + 7) / 8;
    return 8u * (unsigned)a.chunk;
}

// ---------------------------------------------------------------------------
// k_tile
// ---------------------------------------------------------------------------
// A block advances a TX x TY tile by `levels` <= TMAX steps.  Level l pulls
// from level l - 1 and collides on the tile and a halo of M (levels - l)
// nodes (M = the stencil's reach); level 0 is the lattice in HBM, the levels
// between share one LDS buffer of the first level's region, where every node
// keeps its place: a thread pulls its nodes into registers, the block meets,
// and the results overwrite the buffer.  `first`: the run's first step, level
// 1 collides the canonical state S_0 of its own node instead of pulling.
// 64^2 FP64, eight steps: 9 to 10 us on 64 of 256 CUs, whose waves wait 54 % of
// their cycles at the two barriers of a level and for LDS; the vector ALU issues
// a quarter of the time.
struct TileArgs {
    int levels;
    int tiles_x, tiles, chunk;
    int first;
    WallArgs wall;
    MeiStop mei;  // COLL == 3: the iterative initialization's stop
};

template <int QID, class ST, int TX, int TY, int TMAX, int NT>
struct TileShape {
    static constexpr int H = QT<QID>::MAXC * (TMAX - 1);
    static constexpr int W = TX + 2 * H, N = W * (TY + 2 * H);
    static constexpr int K = (N + NT - 1) / NT;  // nodes per thread
};

template <int QID, int COLL, class ST, int TX, int TY, int TMAX, int NT, bool BC, bool ALL>
__device__ __forceinline__ void
tile_region(const typename ST::store_t *__restrict__ C, typename ST::store_t *__restrict__ Cn,
            const StepParams<typename ST::T> &p, const MultiConsts<typename ST::T> &mc,
            const TileArgs &a, const LevelOut *all) {
    using T = typename ST::T;
    using S = typename ST::store_t;
    using SH = TileShape<QID, ST, TX, TY, TMAX, NT>;
    constexpr int Q = QT<QID>::Q, M = QT<QID>::MAXC, W = SH::W, N = SH::N, K = SH::K;
    static_assert(M == 1 && !ST::kNeq, "one-speed stencils, one value per population");
    __shared__ T buf[Q * N];
    if constexpr (COLL == 3)
        if (a.mei.watch && mei_done(a.mei)) return;
    const int tile = tile_of_block(a);
    if (tile >= a.tiles) return;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
    int at[K], xs[K], ys[K], ring[K];
    unsigned bcm[K];
    bool mine[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int n = (int)threadIdx.x + k * NT;
        const int hy = n / W, hx = n - hy * W;
        at[k] = n;
        const int ux = tx * TX - SH::H + hx, uy = ty * TY - SH::H + hy;
        xs[k] = wrap(ux, p.nx);
        ys[k] = wrap(uy, p.ny);
        bcm[k] = BC ? bc_mask<QID>(p, p.bcs, a.wall.walls, xs[k], ys[k]) : 0u;
        // distance outside the tile (0 inside): level l needs ring <= levels - l
        const int dx = max(SH::H - hx, hx - (SH::H + TX - 1)), dy = max(SH::H - hy, hy - (SH::H + TY - 1));
        ring[k] = n < N ? max(0, max(dx, dy)) : TMAX;
        mine[k] = ring[k] == 0 && ux < p.nx && uy < p.ny;
    }
    const int L = a.levels;
    T f[K][Q];
    // the prescribed velocity's part of the equilibrium, read once for all levels
    T pre[COLL == 3 ? K : 1][COLL == 3 ? Q : 1];
    if constexpr (COLL == 3) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (ring[k] > L - 1) continue;
            auto ld = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                pre[k][i] = p.mei[p.plane * i + (long long)xs[k] + (long long)p.nx * ys[k]];
            };
            adj_each_node<QID>(ld);
        }
    }
    // level l's collision of node k, whose state is S_(step + l - 1)
    auto collide = [&](int k, int l) {
        if constexpr (COLL == 3) {
            if (a.mei.watch && mine[k] && xs[k] == p.nx - 1 && ys[k] == p.ny - 1)
                mei_check<QID>(a.mei, f[k], a.mei.step + l - 1);
            const T rho = mei_density<QID>(f[k], LBM_SEQ);
            auto one = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                const T feq = p.w[i] * rho + pre[k][i];
                f[k][i] = p.omo * f[k][i] + p.om * feq;
            };
            adj_each_node<QID>(one);
        } else {
            collide_multi<QID, COLL, ST, T>(f[k], p, mc, xs[k], ys[k]);
        }
    };
    auto store = [&](S *dst, int k) {
        if (!mine[k] || (ALL && !dst)) return;
        auto st = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            dst[p.plane * i + ((long long)xs[k] + (long long)p.nx * ys[k])] = ST::encode(f[k][i], i, p);
        };
        adj_each_node<QID>(st);
    };
    // level 1 from HBM
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (ring[k] > L - 1) continue;
        const int x = xs[k], y = ys[k];
        int xm = x, xp = x, ym = y, yp = y;
        if (!a.first) {
            xm = x == 0 ? p.nx - 1 : x - 1;
            xp = x == p.nx - 1 ? 0 : x + 1;
            ym = y == 0 ? p.ny - 1 : y - 1;
            yp = y == p.ny - 1 ? 0 : y + 1;
        }
        auto ld = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
            const int sx = cx == 0 ? x : (cx > 0 ? xm : xp), sy = cy == 0 ? y : (cy > 0 ? ym : yp);
            f[k][i] = ST::decode(C[p.plane * i + ((long long)sx + (long long)p.nx * sy)], i, p);
        };
        adj_each_node<QID>(ld);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (ring[k] > L - 1) continue;
        if constexpr (BC) {
            if (!a.first)
                bc_apply<QID, T>(p, a.wall.moving, bcm[k], f[k], [&](auto Jc) {
                    return ld_pop<QID, decltype(Jc)::value, ST>(
                        C, p, (long long)xs[k] + (long long)p.nx * ys[k]);
                });
        }
        collide(k, 1);
        if constexpr (ALL) store(static_cast<S *>(all->out[0]), k);
    }
    for (int l = 2; l <= L; ++l) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (ring[k] > L - l + 1) continue;
            auto put = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                buf[N * i + at[k]] = f[k][i];
            };
            adj_each_node<QID>(put);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (ring[k] > L - l) continue;
            auto pull = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                f[k][i] = buf[N * i + at[k] - QT<QID>::cx(i) - W * QT<QID>::cy(i)];
            };
            adj_each_node<QID>(pull);
            if constexpr (BC) {
                bc_apply<QID, T>(p, a.wall.moving, bcm[k], f[k],
                                 [&](auto Jc) { return buf[N * decltype(Jc)::value + at[k]]; });
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (ring[k] > L - l) continue;
            collide(k, l);
            if constexpr (ALL) store(static_cast<S *>(all->out[l - 1]), k);
        }
    }
    if constexpr (!ALL) {
#pragma unroll
        for (int k = 0; k < K; ++k) store(Cn, k);
    }
}

template <int QID, int COLL, class ST, int TX, int TY, int TMAX, int NT, bool BC>
__global__ void __launch_bounds__(NT)
k_tile(const typename ST::store_t *__restrict__ C, typename ST::store_t *__restrict__ Cn,
       const StepParams<typename ST::T> p, const MultiConsts<typename ST::T> mc, const TileArgs a) {
    tile_region<QID, COLL, ST, TX, TY, TMAX, NT, BC, false>(C, Cn, p, mc, a, nullptr);
}

// every level's field kept (k_block_all)
template <int QID, int COLL, class ST, int TX, int TY, int TMAX, int NT>
__global__ void __launch_bounds__(NT)
k_tile_all(const typename ST::store_t *__restrict__ C, const LevelOut o,
           const StepParams<typename ST::T> p, const MultiConsts<typename ST::T> mc,
           const TileArgs a) {
    tile_region<QID, COLL, ST, TX, TY, TMAX, NT, false, true>(C, nullptr, p, mc, a, &o);
}

// x-shift inside a wave: the value of the lane below (D = +1) or above (-1)
template <int D>
__device__ __forceinline__ int lane_shift(int v) {
    // DPP wave_shr:1 / wave_shl:1
    return __builtin_amdgcn_update_dpp(0, v, D > 0 ? 0x138 : 0x130, 0xf, 0xf, true);
}
template <int D>
__device__ __forceinline__ float lane_shift(float v) {
    return __int_as_float(lane_shift<D>(__float_as_int(v)));
}
template <int D>
__device__ __forceinline__ double lane_shift(double v) {
    return __hiloint2double(lane_shift<D>(__double2hiint(v)), lane_shift<D>(__double2loint(v)));
}

// ---------------------------------------------------------------------------
// k_block
// ---------------------------------------------------------------------------
// A block of NW waves advances a region of 64 columns and NW R rows held in
// registers: wave w keeps R consecutive rows, one column per lane.  A pull
// along x comes from the neighbour lane, along y from the wave's own rows, and
// at a wave's first and last row from the neighbouring wave through LDS (two
// buffers, one barrier per level).  Every level computes the whole region; its
// outermost ring of valid nodes is lost each time, so T levels write the inner
// 64 - 2 (T - 1) columns and NW R - 2 (T - 1) rows.
// 1024^2 FP64, five steps: 57 us for 158 MB, the vector ALU issuing 63 % of the
// time; 1021 x 517 FP32, six steps: 22 us in 456 blocks of 16 waves, 60 %, the
// waves waiting 44 % of their cycles, at the levels' barriers above all.
struct BlockArgs {
    int levels;
    int tiles_x, tiles, chunk;
    int outx, outy;  // nodes written per block
    int first;
    WallArgs wall;
};

// the c_y != 0 populations of a wave's boundary rows, in LDS
template <int QID>
LBM_HD constexpr int edge_slot(int i) {
    int n = 0;
    for (int j = 0; j < i; ++j) n += QT<QID>::cy(j) != 0 ? 1 : 0;
    return n;
}
// [buffer][wave][population][column]
template <int QID, class V, int NW>
using BlockEdges = V[2][NW][edge_slot<QID>(QT<QID>::Q)][66];

// One block's region: writes the outx x outy nodes from (cx0, cy0) of a lattice
// of p.nx x p.ny nodes with rows `pitch` apart.
template <int QID, int COLL, class ST, int NW, int R, bool BC, bool ALL = false>
__device__ __forceinline__ void
block_region(const typename ST::store_t *__restrict__ C, typename ST::store_t *__restrict__ Cn,
             const StepParams<typename ST::T> &p, const MultiConsts<typename ST::T> &mc, int pitch,
             int cx0, int cy0, int outx, int outy, int L, int first, WallArgs wall,
             BlockEdges<QID, typename ST::T, NW> &xch, const LevelOut *all = nullptr) {
    using V = typename ST::T;
    using S = typename ST::store_t;
    constexpr int Q = QT<QID>::Q;
    static_assert(QT<QID>::MAXC == 1 && !ST::kNeq, "one-speed stencils, one value per population");
    constexpr int ES = edge_slot<QID>(Q);
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = L - 1;
    const int ux = cx0 - h + lane;
    const int x = wrap(ux, p.nx);
    const int xm = first ? x : (x == 0 ? p.nx - 1 : x - 1);
    const int xp = first ? x : (x == p.nx - 1 ? 0 : x + 1);
    const unsigned off = (unsigned)x * (unsigned)sizeof(S);
    const unsigned offm = (unsigned)xm * (unsigned)sizeof(S), offp = (unsigned)xp * (unsigned)sizeof(S);
    const int row0 = w * R;  // the wave's first row in the region
    int ys[R];
#pragma unroll
    for (int j = 0; j < R; ++j)
        ys[j] = __builtin_amdgcn_readfirstlane(wrap(cy0 - h + row0 + j, p.ny));
    unsigned bcm[R];
#pragma unroll
    for (int j = 0; j < R; ++j) bcm[j] = BC ? bc_mask<QID>(p, p.bcs, wall.walls, x, ys[j]) : 0u;
    V g[R][Q];
    const bool mine_x = ux >= cx0 && ux < min(cx0 + outx, p.nx);
    // row j of a level to `dst`, where this block owns it
    auto store = [&](S *dst, int j, const V(&f)[Q]) {
        const int uy = cy0 - h + row0 + j;
        if (mine_x && uy >= cy0 && uy < min(cy0 + outy, p.ny) && (!ALL || dst)) {
            S *base = dst + (long long)pitch * uy;
            auto st = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                *at_b(base + p.plane * i, off) = ST::encode(f[i], i, p);
            };
            adj_each_node<QID>(st);
        }
    };
    // level 1
    S pre[R][Q];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int y = ys[j];
        const int ym = first ? y : (y == 0 ? p.ny - 1 : y - 1);
        const int yp = first ? y : (y + 1 == p.ny ? 0 : y + 1);
        auto one = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
            const S *base = C + p.plane * i + (long long)pitch * (cy == 0 ? y : (cy > 0 ? ym : yp));
            pre[j][i] = ld_g(at_b(base, cx == 0 ? off : (cx > 0 ? offm : offp)));
        };
        adj_each_node<QID>(one);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int y = ys[j];
        auto dec = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            g[j][i] = ST::decode(pre[j][i], i, p);
        };
        adj_each_node<QID>(dec);
        if constexpr (BC) {
            if (!first)
                bc_apply<QID, V>(p, wall.moving, bcm[j], g[j], [&](auto Jc) {
                    return ld_pop<QID, decltype(Jc)::value, ST>(C, p, (long long)x + (long long)p.nx * y);
                });
        }
        collide_multi<QID, COLL, ST, V>(g[j], p, mc, x, y);
        if constexpr (ALL) store(static_cast<S *>(all->out[0]), j, g[j]);
    }
    for (int l = 2; l <= L; ++l) {
        V(*X)[ES][66] = xch[l & 1];
        auto put = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value, cy = QT<QID>::cy(i);
            if constexpr (cy > 0) X[w][edge_slot<QID>(i)][lane + 1] = g[R - 1][i];
            if constexpr (cy < 0) X[w][edge_slot<QID>(i)][lane + 1] = g[0][i];
        };
        adj_each_node<QID>(put);
        __syncthreads();
        V carry[Q];  // c_y > 0 populations of the row below, already shifted along x
        auto below = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value, cy = QT<QID>::cy(i);
            if constexpr (cy > 0) carry[i] = X[w > 0 ? w - 1 : 0][edge_slot<QID>(i)][lane + 1 - QT<QID>::cx(i)];
        };
        adj_each_node<QID>(below);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int y = ys[j];
            V f[Q];
            auto pull = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
                auto sh = [&](V v) -> V {
                    if constexpr (cx > 0) return lane_shift<1>(v);
                    else if constexpr (cx < 0) return lane_shift<-1>(v);
                    else return v;
                };
                if constexpr (cy > 0) {
                    f[i] = carry[i];
                    carry[i] = sh(g[j][i]);
                } else if constexpr (cy == 0) {
                    f[i] = sh(g[j][i]);
                } else {
                    if (j + 1 < R) f[i] = sh(g[j + 1 < R ? j + 1 : j][i]);
                    else f[i] = X[w + 1 < NW ? w + 1 : w][edge_slot<QID>(i)][lane + 1 - cx];
                }
            };
            adj_each_node<QID>(pull);
            if constexpr (BC) {
                bc_apply<QID, V>(p, wall.moving, bcm[j], f,
                                 [&](auto Jc) { return g[j][decltype(Jc)::value]; });
            }
            collide_multi<QID, COLL, ST, V>(f, p, mc, x, y);
            auto cp = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                g[j][i] = f[i];
            };
            adj_each_node<QID>(cp);
            if constexpr (ALL) store(static_cast<S *>(all->out[l - 1]), j, g[j]);
        }
    }
    if constexpr (!ALL) {
#pragma unroll
        for (int j = 0; j < R; ++j) store(Cn, j, g[j]);
    }
}

template <int QID, int COLL, class ST, int NW, int R, bool BC>
__global__ void __launch_bounds__(64 * NW)
k_block(const typename ST::store_t *__restrict__ C, typename ST::store_t *__restrict__ Cn,
        const StepParams<typename ST::T> p, const MultiConsts<typename ST::T> mc,
        const BlockArgs a) {
    __shared__ BlockEdges<QID, typename ST::T, NW> xch;
    const int tile = tile_of_block(a);
    if (tile >= a.tiles) return;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
    block_region<QID, COLL, ST, NW, R, BC>(C, Cn, p, mc, p.nx, tx * a.outx, ty * a.outy, a.outx,
                                           a.outy, a.levels, a.first, a.wall, xch);
}

// Every level's field kept (the reverse pass needs each step's state): a pass
// reads the lattice once and writes it once per step, where single steps read
// it at each.
template <int QID, int COLL, class ST, int NW, int R>
__global__ void __launch_bounds__(64 * NW)
k_block_all(const typename ST::store_t *__restrict__ C, const LevelOut o,
            const StepParams<typename ST::T> p, const MultiConsts<typename ST::T> mc,
            const BlockArgs a) {
    __shared__ BlockEdges<QID, typename ST::T, NW> xch;
    const int tile = tile_of_block(a);
    if (tile >= a.tiles) return;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
    block_region<QID, COLL, ST, NW, R, false, true>(C, nullptr, p, mc, p.nx, tx * a.outx,
                                                    ty * a.outy, a.outx, a.outy, a.levels, a.first,
                                                    a.wall, xch, &o);
}

// Batched lattices: one region per block from a table; the lattice record is
// read in place with a wave-uniform index (scalar loads).  Bound by FP
// arithmetic (the vector ALU issues 87 % of the time, 48 lattices of 32^2 ..
// 512^2 in FP32); 512 lattices of 200 x 200, us a step against the
// single-step kernel's: 194 / 510 in FP64, 90 / 303 in FP32 (single steps are
// bound by the passes over the pool, 2.9 and 2.4 TB/s there).
template <int QID, int COLL, class ST, int NW, int R>
__global__ void __launch_bounds__(64 * NW)
k_batch_block(const BatchLattice *__restrict__ lats, const BatchRegion *__restrict__ regions,
              int nregions, int chunk, typename ST::store_t *__restrict__ pool, int parity,
              int levels, int first, const StepParams<typename ST::T> base,
              const MultiConsts<typename ST::T> base_mc) {
    using T = typename ST::T;
    __shared__ BlockEdges<QID, T, NW> xch;
    const int r = (int)(blockIdx.x & 7) * chunk + (int)(blockIdx.x >> 3);  // as tile_of_block
    if (r >= nregions) return;
    const BatchRegion g = regions[r];
    const BatchLattice &lat = lats[__builtin_amdgcn_readfirstlane(g.lat)];
    StepParams<T> p = base;
    p.nx = lat.nx;
    p.ny = lat.ny;
    p.plane = lat.plane;
    p.omo = static_cast<T>(lat.omo);
    p.om = static_cast<T>(lat.om);
    p.oms = static_cast<T>(lat.oms);
    p.oma = static_cast<T>(lat.oma);
    MultiConsts<T> mc = base_mc;
    mc.homs = T(0.5) * p.oms;
    mc.homa = T(0.5) * p.oma;
    block_region<QID, COLL, ST, NW, R, false>(pool + lat.off[parity], pool + lat.off[parity ^ 1], p,
                                              mc, lat.pitch, g.x0, g.y0, g.outx, g.outy, levels,
                                              first, WallArgs{0, 0}, xch);
}

// ---------------------------------------------------------------------------
// k_march
// ---------------------------------------------------------------------------
struct MarchArgs {
    int strips, chunks, rows;  // strips of columns, chunks of `rows` rows
    int first;                 // the first level collides S_0 in place
    WallArgs wall;
};

// Geometry of the marching kernel.  A wave holds 64 NC columns, NC adjacent
// ones per lane.  SHIFTED: level 1 pulls straight from HBM (its neighbours
// come from other addresses), so the halo is T - 1 columns; otherwise level 0
// is loaded unshifted, decoded, and is itself a kept level.
template <int QID, class ST, int T, int NC, bool BC>
struct MarchShape {
    static constexpr bool SHIFTED = NC == 1 && !ST::kNeq;
    static constexpr int LINES = SHIFTED ? T - 1 : T;  // levels whose rows are kept
    static constexpr int COLS = 64 * NC;
    static constexpr int HX = (LINES + NC - 1) / NC * NC;  // halo columns, whole lanes
    // columns written, in groups of 64 bytes: where the rows are whole lines a
    // strip's stores then end on memory-transaction boundaries
    static constexpr int GROUP = 64 / (int)sizeof(typename ST::store_t);
    static constexpr int OUT = (COLS - 2 * HX) / GROUP * GROUP;
    static_assert(OUT > 0, "halo wider than the wave");
    // LDS rows of population i per kept level
    LBM_HD static constexpr int slots(int i) {
        if (QT<QID>::cx(i) == 0) return 0;
        return QT<QID>::cy(i) > 0 ? 2 : (QT<QID>::cy(i) == 0 ? 1 : (BC ? 1 : 0));
    }
    LBM_HD static constexpr int slot0(int i) {
        int n = 0;
        for (int j = 0; j < i; ++j) n += slots(j);
        return n;
    }
    static constexpr int LINE = slot0(QT<QID>::Q);  // slots per kept level
};

// 4096^2, a pass: FP64 five steps 2.81 GB (1.16 times one read and one write) at
// 4.2 TB/s, the vector ALU issuing 74 % of the time: either alone would take
// two thirds to three quarters of it, and the waves of the one resident round
// end at different times (1.9 of 3 a SIMD on average).  FP32 six steps 1.57 GB,
// FP16-NEQ four steps 1.05 GB: the ALU issues all the time (91 % and more).
//
// The kept rows of a level, y - 1 (and y - 2 for the populations that moved
// up), while row y arrives: populations with c_x = 0 in registers (they are
// read by the same lane), the others in the wave's own LDS, where the reader
// takes its neighbour's value.  No barrier: a wave's LDS operations execute in
// order.
template <int QID, int COLL, class ST, int T, int NC, bool BC>
__global__ void __launch_bounds__(256)
k_march(const typename ST::store_t *__restrict__ C, typename ST::store_t *__restrict__ Cn,
        const StepParams<typename ST::T> p, const MultiConsts<typename ST::T> mc,
        const MarchArgs a) {
    using V = typename ST::T;
    using S = typename ST::store_t;
    using SH = MarchShape<QID, ST, T, NC, BC>;
    constexpr int Q = QT<QID>::Q, COLS = SH::COLS + 2 * NC, LINES = SH::LINES;
    static_assert(QT<QID>::MAXC == 1, "one-speed stencils");
    __shared__ V rows[4][LINES][SH::LINE][COLS];
    // The boundary list: a row that walks it must not wait for the next row's
    // loads and the stores in flight, as reads of memory would.
    __shared__ BCDev list[BC ? kMaxBC : 1];
    if constexpr (BC) {
        if ((int)threadIdx.x < p.nbc) list[threadIdx.x] = p.bcs[threadIdx.x];
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wave = (int)blockIdx.x * 4 + wv;
    if (wave >= a.strips * a.chunks) return;
    const int chunk = wave / a.strips, strip = wave - chunk * a.strips;
    const int y0 = chunk * a.rows, y1 = min(y0 + a.rows, p.ny);
    const int xo = strip * SH::OUT;           // first column written
    const int col = xo - SH::HX + lane * NC;  // the lane's first column, unwrapped
    const bool out = col >= xo && col < min(xo + SH::OUT, p.nx);
    int xs[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) xs[c] = wrap(col + c, p.nx);
    const bool pulls = SH::SHIFTED && !a.first;
    const int xm = pulls ? (xs[0] == 0 ? p.nx - 1 : xs[0] - 1) : xs[0];
    const int xp = pulls ? (xs[0] == p.nx - 1 ? 0 : xs[0] + 1) : xs[0];
    const unsigned off = (unsigned)xs[0] * (unsigned)sizeof(S);
    const unsigned offm = (unsigned)xm * (unsigned)sizeof(S), offp = (unsigned)xp * (unsigned)sizeof(S);
    // LDS element of the lane's first column and of its neighbours' (rows are
    // padded by NC at both ends: what the end lanes read there is halo)
    const int e0 = lane * NC + NC, em = e0 - 1, ep = e0 + 1;
    // A column's mask changes from row to row only where the lattice or a
    // condition's range begins or ends: it is formed there (row mask_next, and
    // row 0) and kept in between.  Formed at every row, an east or west column
    // held its wave up by some 4,000 cycles a row.
    int mask_next = -1;
    unsigned mask[NC];
    auto masks = [&](int y) {
#pragma unroll
        for (int c = 0; c < NC; ++c) mask[c] = bc_mask<QID>(p, list, a.wall.walls, xs[c], y);
        int next = y < 1 ? 1 : (y < p.ny - 1 ? p.ny - 1 : p.ny);
        for (int b = 0; b < p.nbc; ++b) {
            const int lo = list[b].y0, hi = list[b].y1 + 1;
            if (lo > y && lo < next) next = lo;
            if (hi > y && hi < next) next = hi;
        }
        mask_next = __builtin_amdgcn_readfirstlane(next);
    };
    // boundary masks of the row each level holds: they move down with the rows
    unsigned bcm[LINES + 1][NC];
#pragma unroll
    for (int l = 0; l <= LINES; ++l)
#pragma unroll
        for (int c = 0; c < NC; ++c) bcm[l][c] = 0u;
    V mid[LINES][NC][Q], up[LINES][NC][Q];  // c_x = 0 only
#pragma unroll
    for (int l = 0; l < LINES; ++l)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < Q; ++i) mid[l][c][i] = up[l][c][i] = V(0);
    int r = __builtin_amdgcn_readfirstlane(wrap(y0 - LINES, p.ny));  // row of the first level
    Pack<S, NC> pre[Q];
    Pack<Rec16, NC> rec;
    auto fetch = [&](int row) {
        const int rm = !pulls ? row : (row == 0 ? p.ny - 1 : row - 1);
        const int rp = !pulls ? row : (row + 1 == p.ny ? 0 : row + 1);
        if constexpr (ST::kNeq)
            rec = ld_g(at_b(reinterpret_cast<const Pack<Rec16, NC> *>(ST::recs(C) + (long long)p.nx * row),
                            off * (unsigned)(sizeof(Rec16) / sizeof(S))));
        auto one = [&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
            const int rs = cy == 0 ? row : (cy > 0 ? rm : rp);
            const S *plane0 = C;
            if constexpr (ST::kNeq) plane0 = ST::pops(C, p.plane);
            const S *base = plane0 + p.plane * i + (long long)p.nx * rs;
            const unsigned o = cx == 0 ? off : (cx > 0 ? offm : offp);
            pre[i] = ld_g(at_b(reinterpret_cast<const Pack<S, NC> *>(base), o));
        };
        adj_each_node<QID>(one);
    };
    fetch(r);
    const int iters = (y1 - y0) + 2 * LINES;
#pragma unroll 1
    for (int k = 0; k < iters; ++k) {
        V n[NC][Q];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if constexpr (ST::kNeq) {
                const Mom4 m = ST::unpack(rec.v[c]);
                auto dec = [&](auto Ic) {
                    constexpr int i = decltype(Ic)::value;
                    n[c][i] = geq_rec<QID, i>(m, p) + ST::to_f(pre[i].v[c], p);
                };
                adj_each_node<QID>(dec);
            } else {
                auto dec = [&](auto Ic) {
                    constexpr int i = decltype(Ic)::value;
                    n[c][i] = ST::decode(pre[i].v[c], i, p);
                };
                adj_each_node<QID>(dec);
            }
        }
        int rl = r;  // the row of the level in hand
        r = __builtin_amdgcn_readfirstlane(r + 1 == p.ny ? 0 : r + 1);
        if (k + 1 < iters) fetch(r);
        if constexpr (BC) {
            if (k == 0 || rl == 0 || rl == mask_next) masks(rl);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
#pragma unroll
                for (int l = LINES; l > 0; --l) bcm[l][c] = bcm[l - 1][c];
                bcm[0][c] = mask[c];
            }
        }
        if (SH::SHIFTED || a.first) {
            if constexpr (BC && SH::SHIFTED) {
                if (!a.first)
                    bc_apply<QID, V>(p, a.wall.moving, bcm[0][0], n[0], [&](auto Jc) {
                        return ld_pop<QID, decltype(Jc)::value, ST>(
                            C, p, (long long)xs[0] + (long long)p.nx * rl);
                    });
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) collide_multi<QID, COLL, ST, V>(n[c], p, mc, xs[c], rl);
        }
        const int par = k & 1;
        Rec16 orec[NC];
        float nq[NC][Q];
        // the next level at row y - 1 from level l's rows y - 2, y - 1, y
        auto level = [&](auto Lc) {
            constexpr int l = decltype(Lc)::value;
            rl = __builtin_amdgcn_readfirstlane(rl == 0 ? p.ny - 1 : rl - 1);
            V(*L)[COLS] = rows[wv][l];
            V f[NC][Q];
            auto pull = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i), s0 = SH::slot0(i);
                if constexpr (cx == 0) {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        f[c][i] = cy > 0 ? up[l][c][i] : (cy == 0 ? mid[l][c][i] : n[c][i]);
                } else if constexpr (cy < 0) {
                    if constexpr (cx > 0) {
#pragma unroll
                        for (int c = NC - 1; c > 0; --c) f[c][i] = n[c - 1][i];
                        f[0][i] = lane_shift<1>(n[NC - 1][i]);
                    } else {
#pragma unroll
                        for (int c = 0; c + 1 < NC; ++c) f[c][i] = n[c + 1][i];
                        f[NC - 1][i] = lane_shift<-1>(n[0][i]);
                    }
                } else {
                    const V *src = cy > 0 ? L[s0 + par] : L[s0];
#pragma unroll
                    for (int c = 0; c < NC; ++c) f[c][i] = src[(cx > 0 ? em : ep) + c];
                }
            };
            adj_each_node<QID>(pull);
            if constexpr (BC) {
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    bc_apply<QID, V>(p, a.wall.moving, bcm[l + 1][c], f[c], [&](auto Jc) {
                        constexpr int j = decltype(Jc)::value;
                        constexpr int s0 = SH::slot0(j);
                        if constexpr (QT<QID>::cx(j) == 0) return mid[l][c][j];
                        else if constexpr (QT<QID>::cy(j) > 0) return L[s0 + (par ^ 1)][e0 + c];
                        else return L[s0][e0 + c];
                    });
            }
            // the rows move down; the compiler must not reorder the lane's own
            // LDS accesses (neighbour lanes read what this lane wrote)
            asm volatile("" ::: "memory");
            auto keep = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i), s0 = SH::slot0(i);
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    if constexpr (cx == 0) {
                        if constexpr (cy > 0) up[l][c][i] = mid[l][c][i];
                        mid[l][c][i] = n[c][i];
                    } else if constexpr (cy > 0) {
                        L[s0 + par][e0 + c] = n[c][i];
                    } else if constexpr (cy == 0 || BC) {
                        L[s0][e0 + c] = n[c][i];
                    }
                }
            };
            adj_each_node<QID>(keep);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if constexpr (ST::kNeq) {
                    if constexpr (l == LINES - 1) {
                        collide_neq<QID, COLL, ST>(f[c], p, xs[c], rl, orec[c], nq[c], LBM_SEQ);
                        continue;
                    }
                }
                collide_multi<QID, COLL, ST, V>(f[c], p, mc, xs[c], rl);
                auto cp = [&](auto Ic) {
                    constexpr int i = decltype(Ic)::value;
                    n[c][i] = f[c][i];
                };
                adj_each_node<QID>(cp);
            }
        };
        mrt_each(level, std::make_integer_sequence<int, LINES>{});
        if (k >= 2 * LINES && out) {
            if constexpr (ST::kNeq) {
                Pack<Rec16, NC> pr;
#pragma unroll
                for (int c = 0; c < NC; ++c) pr.v[c] = orec[c];
                Pack<Pack<Rec16, NC>, 1> pm;
                pm.v[0] = pr;
                put_pack<true>(at_b(reinterpret_cast<Pack<Rec16, NC> *>(ST::recs(Cn) + (long long)p.nx * rl),
                                    off * (unsigned)(sizeof(Rec16) / sizeof(S))), pm);
            }
            auto st = [&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                S *plane0 = Cn;
                if constexpr (ST::kNeq) plane0 = ST::pops(Cn, p.plane);
                Pack<S, NC> pk;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    if constexpr (ST::kNeq) pk.v[c] = ST::raw(nq[c][i]);
                    else pk.v[c] = ST::encode(n[c][i], i, p);
                }
                Pack<Pack<S, NC>, 1> pm;
                pm.v[0] = pk;
                put_pack<true>(at_b(reinterpret_cast<Pack<S, NC> *>(plane0 + p.plane * i + (long long)p.nx * rl), off), pm);
            };
            adj_each_node<QID>(st);
        }
    }
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
constexpr int kTileX = 8, kTileY = 8, kTileT = 8, kTileThreads = 512;

template <class T>
TileArgs tile_args(const MultiLaunch &L, const StepParams<T> &p, unsigned &blocks) {
    TileArgs a;
    a.levels = L.steps;
    a.first = L.first;
    a.wall = WallArgs{L.walls, L.moving};
    a.mei = L.mei;
    a.tiles_x = (p.nx + kTileX - 1) / kTileX;
    blocks = deal_tiles(a, (p.ny + kTileY - 1) / kTileY);
    return a;
}

template <int QID, int COLL, class ST, bool BC>
int launch_tile(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    using S = typename ST::store_t;
    if (L.steps < 1 || L.steps > kTileT) return -5;
    unsigned blocks;
    const TileArgs a = tile_args(L, p, blocks);
    k_tile<QID, COLL, ST, kTileX, kTileY, kTileT, kTileThreads, BC><<<blocks, kTileThreads, 0, s>>>(
        static_cast<const S *>(L.src), static_cast<S *>(L.dst), p, multi_consts(p), a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <class S, int ROWS, class T>
BlockArgs block_args(const MultiLaunch &L, const StepParams<T> &p, unsigned &blocks) {
    BlockArgs a;
    a.levels = L.steps;
    a.first = L.first;
    a.wall = WallArgs{L.walls, L.moving};
    const BlockShape b = block_shape(p.nx, p.ny, L.steps, ROWS, (int)sizeof(S));
    a.outx = b.outx;
    a.outy = b.outy;
    a.tiles_x = b.across;
    blocks = deal_tiles(a, b.down);
    return a;
}
// the output of a block is at least two rows and two columns
constexpr bool block_fits(int steps, int rows) {
    return steps >= 1 && 2 * (steps - 1) < 64 && 2 * (steps - 1) < rows;
}

template <int QID, int COLL, class ST, int NW, int R, bool BC>
int launch_block(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    using S = typename ST::store_t;
    if (!block_fits(L.steps, NW * R)) return -5;
    unsigned blocks;
    const BlockArgs a = block_args<S, NW * R>(L, p, blocks);
    k_block<QID, COLL, ST, NW, R, BC><<<blocks, 64 * NW, 0, s>>>(
        static_cast<const S *>(L.src), static_cast<S *>(L.dst), p, multi_consts(p), a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// every step's field kept, periodic SRT/TRT lattices
template <int QID, int COLL, class ST, int NW, int R>
int launch_block_all(const MultiLaunch &L, const LevelOut &o, const StepParams<typename ST::T> &p,
                     hipStream_t s) {
    using S = typename ST::store_t;
    if (!block_fits(L.steps, NW * R) || L.steps > 8) return -5;
    unsigned blocks;
    const BlockArgs a = block_args<S, NW * R>(L, p, blocks);
    k_block_all<QID, COLL, ST, NW, R><<<blocks, 64 * NW, 0, s>>>(
        static_cast<const S *>(L.src), o, p, multi_consts(p), a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <int QID, int COLL, class ST>
int launch_all(const MultiLaunch &L, const LevelOut &o, const StepParams<typename ST::T> &p,
               hipStream_t s) {
    using S = typename ST::store_t;
    constexpr bool f64 = sizeof(S) == 8;
    switch (L.kernel) {
    case kMultiTile: {
        if (L.steps < 1 || L.steps > kTileT) return -5;
        unsigned blocks;
        const TileArgs a = tile_args(L, p, blocks);
        k_tile_all<QID, COLL, ST, kTileX, kTileY, kTileT, kTileThreads>
            <<<blocks, kTileThreads, 0, s>>>(static_cast<const S *>(L.src), o, p, multi_consts(p), a);
        return hipGetLastError() == hipSuccess ? 0 : -4;
    }
    case kMultiBlock16: return launch_block_all<QID, COLL, ST, 16, 1>(L, o, p, s);
    case kMultiBlock32: return launch_block_all<QID, COLL, ST, 16, 2>(L, o, p, s);
    case kMultiBlockWide: return launch_block_all<QID, COLL, ST, 8, f64 ? 3 : 4>(L, o, p, s);
    default: return -5;
    }
}

// FP64: the pair form (the same bits as the single-step kernels').  FP32: SRT
// in the single-step kernels' own form, which gives their bits too; TRT has no
// such kernels (see adj_plan).
template <class ST>
int launch_all_any(const MultiLaunch &L, const LevelOut &o, const StepParams<typename ST::T> &p,
                   hipStream_t s) {
    constexpr bool f64 = sizeof(typename ST::store_t) == 8;
    if constexpr (f64)
        switch (L.coll == 1 ? L.qid : 0) {
        case 4: return launch_all<4, 1, ST>(L, o, p, s);
        case 5: return launch_all<5, 1, ST>(L, o, p, s);
        case 9: return launch_all<9, 1, ST>(L, o, p, s);
        }
    constexpr int SRT = f64 ? 0 : 4;
    switch (L.coll == 0 ? L.qid : 0) {
    case 4: return launch_all<4, SRT, ST>(L, o, p, s);
    case 5: return launch_all<5, SRT, ST>(L, o, p, s);
    case 9: return launch_all<9, SRT, ST>(L, o, p, s);
    default: return -1;
    }
}


template <int QID, int COLL, class ST, int T, int NC, bool BC>
int launch_march(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    using S = typename ST::store_t;
    using SH = MarchShape<QID, ST, T, NC, BC>;
    if (p.nx % NC != 0 || p.nx > kMultiMaxNx) return -5;
    static const int slots = [] {
        int per_cu = 0, dev = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, k_march<QID, COLL, ST, T, NC, BC>, 256, 0) != hipSuccess ||
            hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        return per_cu * cus * 4;
    }();
    if (slots < 1) return -4;
    MarchArgs a;
    a.first = L.first;
    a.wall = WallArgs{L.walls, L.moving};
    a.strips = (p.nx + SH::OUT - 1) / SH::OUT;
    // rows per wave: one resident round of waves, at least kMarchRows (the
    // 2 LINES warm-up rows of a chunk are recomputed)
    const long long per_round = ((long long)p.ny * a.strips + slots - 1) / slots;
    a.rows = (int)(per_round > kMarchRows ? per_round : kMarchRows);
    if (a.rows > p.ny) a.rows = p.ny;
    a.chunks = (p.ny + a.rows - 1) / a.rows;
    const long long waves = (long long)a.strips * a.chunks;
    k_march<QID, COLL, ST, T, NC, BC><<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(
        static_cast<const S *>(L.src), static_cast<S *>(L.dst), p, multi_consts(p), a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <int QID, int COLL, class ST, bool BC>
int launch_multi_c(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    if constexpr (ST::kNeq) {
        if (L.kernel != kMultiMarch) return -5;
        // level 0 is decoded in place: a first pass collides it too
        switch (L.steps - L.first) {
        case 1: return launch_march<QID, COLL, ST, 1, 2, BC>(L, p, s);
        case 2: return launch_march<QID, COLL, ST, 2, 2, BC>(L, p, s);
        case 3: return launch_march<QID, COLL, ST, 3, 2, BC>(L, p, s);
        case 4: return launch_march<QID, COLL, ST, 4, 2, BC>(L, p, s);
        default: return -5;
        }
    } else {
        constexpr bool f64 = sizeof(typename ST::store_t) == 8;
        switch (L.kernel) {
        case kMultiTile: return launch_tile<QID, COLL, ST, BC>(L, p, s);
        case kMultiBlock16: return launch_block<QID, COLL, ST, 16, 1, BC>(L, p, s);
        case kMultiBlock32: return launch_block<QID, COLL, ST, 16, 2, BC>(L, p, s);
        case kMultiBlockWide:
            if constexpr (f64) return launch_block<QID, COLL, ST, 8, 3, BC>(L, p, s);
            else return launch_block<QID, COLL, ST, 8, 4, BC>(L, p, s);
        case kMultiMarch: break;
        default: return -5;
        }
        switch (L.steps) {
        case 2: return launch_march<QID, COLL, ST, 2, 1, BC>(L, p, s);
        case 3: return launch_march<QID, COLL, ST, 3, 1, BC>(L, p, s);
        case 4: return launch_march<QID, COLL, ST, 4, 1, BC>(L, p, s);
        case 5: if constexpr (f64) return launch_march<QID, COLL, ST, 5, 1, BC>(L, p, s); break;
        case 6: if constexpr (!f64) return launch_march<QID, COLL, ST, 6, 1, BC>(L, p, s); break;
        default: break;
        }
        return -5;
    }
}

template <int QID, class ST>
int launch_multi(const MultiLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    const bool bc = p.nbc > 0;
    switch (L.coll) {
    case 0: return bc ? launch_multi_c<QID, 0, ST, true>(L, p, s) : launch_multi_c<QID, 0, ST, false>(L, p, s);
    case 1: return bc ? launch_multi_c<QID, 1, ST, true>(L, p, s) : launch_multi_c<QID, 1, ST, false>(L, p, s);
    case 2:
        if constexpr (ST::id == 0)
            return bc ? launch_multi_c<QID, 2, ST, true>(L, p, s)
                      : launch_multi_c<QID, 2, ST, false>(L, p, s);
        break;
    default: break;
    }
    return -2;
}

// Batched lattices: the wide blocks (the region table is cut for the largest
// pass; smaller passes use the same regions)
template <int QID, class ST>
int launch_batch_block(int coll, const BatchLattice *lats, const BatchRegion *regions, int nregions,
                       void *pool, int parity, int levels, int first,
                       const StepParams<typename ST::T> &p, hipStream_t s) {
    using S = typename ST::store_t;
    constexpr int NW = 8, R = sizeof(S) == 8 ? kBatchRowsF64 / NW : kBatchRowsF32 / NW;
    constexpr int tmax = sizeof(S) == 8 ? kBatchStepsF64 : kBatchStepsF32;
    if (levels < 1 || levels > tmax || nregions < 1) return -5;
    S *pl = static_cast<S *>(pool);
    const int chunk = (nregions + 7) / 8;
    const unsigned blocks = 8u * (unsigned)chunk;
    if (coll == 0)
        k_batch_block<QID, 0, ST, NW, R><<<blocks, 64 * NW, 0, s>>>(
            lats, regions, nregions, chunk, pl, parity, levels, first, p, multi_consts(p));
    else
        k_batch_block<QID, 1, ST, NW, R><<<blocks, 64 * NW, 0, s>>>(
            lats, regions, nregions, chunk, pl, parity, levels, first, p, multi_consts(p));
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

#define LBM_DEFINE_BATCH_BLOCK(TAG, ST, QID)                                                     \
    int run_batch_block_##TAG##_q##QID(int coll, const BatchLattice *lats,                       \
                                       const BatchRegion *regions, int nregions, void *pool,     \
                                       int parity, int levels, int first,                        \
                                       const StepParams<typename ST::T> &p, hipStream_t s) {     \
        return launch_batch_block<QID, ST>(coll, lats, regions, nregions, pool, parity, levels,  \
                                           first, p, s);                                         \
    }

// one translation unit per (storage, quadrature)
#define LBM_DEFINE_MULTI(TAG, ST, QID)                                                      \
    int run_multi_##TAG##_q##QID(const MultiLaunch &L, const StepParams<typename ST::T> &p, \
                                 hipStream_t s) {                                           \
        return launch_multi<QID, ST>(L, p, s);                                              \
    }

}  // namespace lbm
