// lbm_adjoint.h -- reverse-mode (adjoint) kernels of the periodic SRT/TRT
// collide-stream step, for gradients of a velocity-field loss.
//
// Forward step t (the reference's collide! then stream!, periodic lattice):
//   C_t[x, i]     = Omega_i(S_t[x, :])                       (per node)
//   S_{t+1}[x, i] = C_t[x - c_i, i]                           (pull stream)
// with S_0 = feq(rho0, u0) and loss L = 1/2 sum_x |u(S_T)[x] - u_target[x]|^2.
// Reverse step, lambda_t = dL/dS_t:
//   mu_t[x, i]     = lambda_{t+1}[x + c_i, i]                 (transposed stream: push)
//   lambda_t[x, :] = J_Omega(S_t[x, :])^T mu_t[x, :]          (per node)
// The collision Jacobian.  With nu_i = om mu_i (SRT) or
// nu_i = om_s mu+_i + om_a mu-_i (TRT, mu+- the (anti)symmetric parts under
// i <-> opp(i)), both operators give
//   (J^T mu)_j = mu_j - nu_j + sum_i nu_i dfeq_i/df_j,
//   sum_i nu_i dfeq_i/df_j = A + B . (c_j - u) / rho,
//   A = sum_i nu_i feq_i / rho,   B_d = sum_i nu_i dfeq_i/du_d,
// since rho = sum f, u = sum c f / rho (so du_d/df_j = (c_jd - u_d)/rho) and
// feq_i = w_i rho P_i(u).  Relaxation-time sensitivities accumulate per node:
//   dL/dtau   += sum_i mu_i (f_i - feq_i) / tau^2                 (SRT)
//   dL/dtau_s += sum_i mu+_i (f_i - feq_i) / tau_s^2, likewise tau_a with mu-.
// Adjoint fields are plain (unshifted) arrays of the arithmetic type in the
// structure-of-arrays layout lam[x + nx*(y + ny*i)].
#pragma once

#include "lbm_multi.h"

namespace lbm {

// d feq_I / d u, for the closed-form equilibria of order FEQ = 1..4 of feq_i
// (the polynomial of maxwell_boltzmann_equilibrium.jl:43-66)
template <int QID, int I, class T>
__device__ __forceinline__ void dfeq_du(T rho, T ux, T uy, T usq, const StepParams<T> &p, T &gx,
                                        T &gy) {
    constexpr int FEQ = QT<QID>::FEQ;
    const T cx = static_cast<T>(QT<QID>::cx(I)), cy = static_cast<T>(QT<QID>::cy(I));
    const T ud = cx * ux + cy * uy;
    // d/du_d of the polynomial = kc * c_d + ku * u_d
    T kc = p.s, ku = T(0);
    if constexpr (FEQ >= 2) {
        kc = kc + p.s2 * ud;
        ku = ku - p.s;
    }
    if constexpr (FEQ >= 3) {
        const T s3 = p.s2 * p.s;
        kc = kc + T(0.5) * (s3 * (ud * ud) - p.s2 * usq);
        ku = ku - p.s2 * ud;
        if constexpr (FEQ >= 4) {
            kc = kc + T(1.0 / 6.0) * (p.s4 * (ud * ud * ud)) - T(0.5) * (s3 * usq * ud);
            ku = ku - T(0.5) * (s3 * (ud * ud)) + T(0.5) * (p.s2 * usq);
        }
    }
    const T wr = p.w[I] * rho;
    gx = wr * (kc * cx + ku * ux);
    gy = wr * (kc * cy + ku * uy);
}

template <int QID, int... Is, class F>
__device__ __forceinline__ void adj_each(F &&fn, std::integer_sequence<int, Is...>) {
    (fn(std::integral_constant<int, Is>{}), ...);
}
#define LBM_ADJ_EACH(...) adj_each<QID>(__VA_ARGS__, LBM_SEQ)

// state S_t of node (x, y): stored directly (DIRECT) or pulled from C_{t-1}
template <int QID, class ST, bool DIRECT>
__device__ __forceinline__ void adj_state(const typename ST::store_t *__restrict__ src,
                                          const StepParams<typename ST::T> &p, int x, int y,
                                          long long n, typename ST::T (&f)[QT<QID>::Q]) {
    if constexpr (DIRECT) load_local<QID, ST>(src, p, n, f, LBM_SEQ);
    else pull_seq<QID, ST>(src, p, x, y, f, LBM_SEQ);
}

// rho, u of a state (the FP32 storages hold g = f - w rho0)
template <int QID, class ST>
__device__ __forceinline__ void adj_moments(const typename ST::T (&f)[QT<QID>::Q],
                                            const StepParams<typename ST::T> &p,
                                            typename ST::T &drho, typename ST::T &rho,
                                            typename ST::T &ux, typename ST::T &uy) {
    if constexpr (ST::kShift) {
        node_moments_dev<QID>(f, p, drho, ux, uy);
        rho = p.rho0 + drho;
    } else {
        node_moments<QID>(f, rho, ux, uy);
        drho = rho - p.rho0;
    }
}

// lambda of a node from its state f and mu: lam = J^T(f) mu; gs, ga: its terms
// of dL/dtau (times the squared rate).  First- and second-order equilibria, one
// opposite pair (i, o) at a time: with ud = u . c_i, q = s^2/2 ud^2 - s/2 u^2,
// feq_i +- feq_o = 2 w rho (1 + q), 2 w rho s ud, and the sums and differences
// of nu give the pair's terms of A and B at once (B is divided by rho, which
// cancels rho in dfeq/du).  D2Q9 SRT FP64: 238 arithmetic instructions instead
// of 339.
template <int QID, class ST, int COLL>
__device__ __forceinline__ void adj_node_pairs(const typename ST::T (&f)[QT<QID>::Q],
                                               const typename ST::T (&mu)[QT<QID>::Q],
                                               const StepParams<typename ST::T> &p,
                                               typename ST::T (&lam)[QT<QID>::Q],
                                               typename ST::T &gs, typename ST::T &ga) {
    using T = typename ST::T;
    constexpr int FEQ = QT<QID>::FEQ;
    static_assert(FEQ <= 2, "first- and second-order equilibria");
    T rho, ux, uy, e0;  // e0: the density as the storage holds it
    if constexpr (ST::kShift) {
        node_moments_dev<QID>(f, p, e0, ux, uy);
        rho = p.rho0 + e0;
    } else {
        moments_div2<QID>(f, rho, ux, uy, LBM_SEQ);
        e0 = rho;
    }
    const T oms = COLL == 0 ? p.om : p.oms, oma = COLL == 0 ? p.om : p.oma;
    const T hs2 = T(0.5) * p.s2, hq = FEQ == 2 ? (T(0.5) * p.s) * (ux * ux + uy * uy) : T(0);
    const T r2 = T(2) * rho, e2 = T(2) * e0;
    T A = T(0), Bx = T(0), By = T(0), M = T(0);
    gs = ga = T(0);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value, o = QT<QID>::opp(i), wr = weight_rep<QID>(i);
        constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
        if constexpr (i == o) {
            const T ap = p.w[wr] * (oms * mu[i]);
            gs = gs + mu[i] * (T(2) * f[i] - p.w[wr] * (e2 - r2 * hq));
            A = A + ap * (T(1) - hq);
            M = M + ap;
        } else if constexpr (i < o) {
            const T ud = udot<QID, i>(ux, uy), ps = p.s * ud;
            const T sp = mu[i] + mu[o], sm = mu[i] - mu[o];
            const T ap = p.w[wr] * (oms * sp), am = p.w[wr] * (oma * sm);
            T q = T(0), k = am * p.s;
            if constexpr (FEQ == 2) {
                q = hs2 * (ud * ud) - hq;
                k = k + ap * (p.s2 * ud);
            }
            const T ns = (f[i] + f[o]) - p.w[wr] * (e2 + r2 * q);
            const T na = (f[i] - f[o]) - p.w[wr] * (r2 * ps);
            gs = gs + sp * ns;
            if constexpr (COLL == 0) gs = gs + sm * na;
            else ga = ga + sm * na;
            A = A + (ap * (T(1) + q) + am * ps);
            M = M + ap;
            if constexpr (cx != 0) Bx = Bx + cmul<cx>(k);
            if constexpr (cy != 0) By = By + cmul<cy>(k);
        }
    });
    gs = T(0.5) * gs;
    ga = T(0.5) * ga;
    if constexpr (FEQ == 2) {
        const T sm = p.s * M;
        Bx = Bx - ux * sm;
        By = By - uy * sm;
    }
    const T base = A - (Bx * ux + By * uy);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value, o = QT<QID>::opp(i);
        if constexpr (i == o) {
            lam[i] = (mu[i] - oms * mu[i]) + base;
        } else if constexpr (i < o) {
            const T bc = udot<QID, i>(Bx, By);
            if constexpr (COLL == 0) {
                lam[i] = (mu[i] - oms * mu[i]) + (base + bc);
                lam[o] = (mu[o] - oms * mu[o]) + (base - bc);
            } else {
                const T np = (T(0.5) * oms) * (mu[i] + mu[o]), nm = (T(0.5) * oma) * (mu[i] - mu[o]);
                lam[i] = (mu[i] - (np + nm)) + (base + bc);
                lam[o] = (mu[o] - (np - nm)) + (base - bc);
            }
        }
    });
}

// the same for any order
template <int QID, class ST, int COLL>
__device__ __forceinline__ void adj_node_sum(const typename ST::T (&f)[QT<QID>::Q],
                                         const typename ST::T (&mu)[QT<QID>::Q],
                                         const StepParams<typename ST::T> &p,
                                         typename ST::T (&lam)[QT<QID>::Q], typename ST::T &gs,
                                         typename ST::T &ga) {
    using T = typename ST::T;
    constexpr int Q = QT<QID>::Q;
    T drho, rho, ux, uy;
    adj_moments<QID, ST>(f, p, drho, rho, ux, uy);
    const T usq = ux * ux + uy * uy;
    T feq[Q], neq[Q];
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        if constexpr (ST::kShift) {
            const T g = feq_dev_i<QID, i, T>(drho, rho, ux, uy, usq, p);
            neq[i] = f[i] - g;
            feq[i] = g + p.w[i] * p.rho0;
        } else {
            feq[i] = feq_i<QID, i, T>(rho, ux, uy, usq, p);
            neq[i] = f[i] - feq[i];
        }
    });
    T nu[Q];
    gs = ga = T(0);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        if constexpr (COLL == 0) {
            nu[i] = p.om * mu[i];
            gs = gs + mu[i] * neq[i];
        } else {
            constexpr int o = QT<QID>::opp(i);
            const T mp = T(0.5) * (mu[i] + mu[o]), mm = T(0.5) * (mu[i] - mu[o]);
            nu[i] = p.oms * mp + p.oma * mm;
            gs = gs + mp * neq[i];
            ga = ga + mm * neq[i];
        }
    });
    T A = T(0), Bx = T(0), By = T(0);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        T gx, gy;
        dfeq_du<QID, i, T>(rho, ux, uy, usq, p, gx, gy);
        A = A + nu[i] * feq[i];
        Bx = Bx + nu[i] * gx;
        By = By + nu[i] * gy;
    });
    const T ir = T(1) / rho;
    A = A * ir;
    Bx = Bx * ir;
    By = By * ir;
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int j = decltype(Ic)::value;
        const T cx = static_cast<T>(QT<QID>::cx(j)), cy = static_cast<T>(QT<QID>::cy(j));
        lam[j] = (mu[j] - nu[j]) + (A + (Bx * (cx - ux) + By * (cy - uy)));
    });
}

// FP32 keeps the plain sums: its dL/dtau moves less with their rounding unchanged
template <int QID, class ST, int COLL>
__device__ __forceinline__ void adj_node(const typename ST::T (&f)[QT<QID>::Q],
                                         const typename ST::T (&mu)[QT<QID>::Q],
                                         const StepParams<typename ST::T> &p,
                                         typename ST::T (&lam)[QT<QID>::Q], typename ST::T &gs,
                                         typename ST::T &ga) {
    if constexpr (QT<QID>::FEQ <= 2 && !ST::kShift) adj_node_pairs<QID, ST, COLL>(f, mu, p, lam, gs, ga);
    else adj_node_sum<QID, ST, COLL>(f, mu, p, lam, gs, ga);
}

// the step's terms of dL/dtau, FP64
template <int COLL, class T>
__device__ __forceinline__ void adj_tau(T gs, T ga, const StepParams<T> &p, double &g0, double &g1) {
    if constexpr (COLL == 0) {
        g0 += static_cast<double>(gs) * (static_cast<double>(p.om) * static_cast<double>(p.om));
    } else {
        g0 += static_cast<double>(gs) * (static_cast<double>(p.oms) * static_cast<double>(p.oms));
        g1 += static_cast<double>(ga) * (static_cast<double>(p.oma) * static_cast<double>(p.oma));
    }
}

// one reverse step: lam = J^T(S_t) mu, mu pushed from lam_next
template <int QID, class ST, int COLL, bool DIRECT>
__global__ void __launch_bounds__(256)
k_adj_step(const typename ST::T *__restrict__ lam_next, const typename ST::store_t *__restrict__ src,
           typename ST::T *__restrict__ lam, double *__restrict__ gtau,
           const StepParams<typename ST::T> p) {
    using T = typename ST::T;
    constexpr int Q = QT<QID>::Q;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= p.nx) return;
    const long long n = (long long)x + (long long)p.nx * y;
    T f[Q];
    adj_state<QID, ST, DIRECT>(src, p, x, y, n, f);
    T mu[Q];
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        const int sx = wrap(x + QT<QID>::cx(i), p.nx), sy = wrap(y + QT<QID>::cy(i), p.ny);
        mu[i] = lam_next[p.plane * i + (long long)sx + (long long)p.nx * sy];
    });
    T out[Q], gs, ga;
    adj_node<QID, ST, COLL>(f, mu, p, out, gs, ga);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int j = decltype(Ic)::value;
        lam[p.plane * j + n] = out[j];
    });
    double unused = 0.0;
    adj_tau<COLL>(gs, ga, p, gtau[n], COLL == 0 ? unused : gtau[p.plane + n]);
}

// Several reverse steps of a one-speed stencil per launch: a block takes a
// 16 x 16 tile of lambda through `levels` steps, level l on the tile and a halo
// of levels - l nodes; lambda stays in LDS, the state of each step is pulled
// from its post-collision field (loaded before the block meets, so that it
// arrives behind the exchange).  A single step reads lambda and the state and
// writes lambda, 27 populations a node; here lambda moves once per launch.
// Same operations in the same order per node and step: in FP64 the bits of
// single steps (FP32: another contraction of products and sums).
// Bound by the pulls of the state (512^2 FP64, launches of three and four steps:
// 103 MB in 26 us, waves waiting 44 % of their cycles, the vector ALU issuing 45 %
// of the time): a tile's 22 columns touch three 128-byte lines a row, so neighbouring tiles share most
// lines and run on one XCD, with one L2 (consecutive workgroups go to the 8 XCDs
// in turn; the tiles are dealt in 8 contiguous chunks).  D2Q9 SRT FP64 / FP32, us
// a step, single steps with
// the plain node sum 12.9 in FP64: single steps 11.3 / 9.6 on 512^2, 5.2 / 4.9
// on 128^2; four steps, tiles dealt in turn 11.0 / 7.5 and 2.5 / 1.7; in chunks
// 7.5 / 4.4 and 2.4 / 1.7.  Two blocks fit a CU (128 registers); 26 x 26 tiles
// of 1024 threads recompute less but fit once (8.1), 8 x 8 tiles recompute more
// (10.7), 26 x 10 tiles read fewer lines a row in more rows (8.5).
constexpr int kAdjTile = 16, kAdjThreads = 512;
struct AdjLevels {
    const void *state[kAdjLevels];  // by level, latest step first
    int levels;
    int direct;  // the last level's state is S_0 itself
    int tiles_x, tiles, chunk;
};

template <int QID, class ST, int COLL>
__global__ void __launch_bounds__(kAdjThreads, 4)
k_adj_tile(const typename ST::T *__restrict__ lam_next, typename ST::T *__restrict__ lam,
           double *__restrict__ gtau, const StepParams<typename ST::T> p, const AdjLevels a) {
    using T = typename ST::T;
    using S = typename ST::store_t;
    constexpr int Q = QT<QID>::Q, H = kAdjLevels - 1, W = kAdjTile + 2 * H, N = W * (kAdjTile + 2 * H);
    static_assert(QT<QID>::MAXC == 1 && !ST::kNeq && N <= kAdjThreads, "one node per thread");
    __shared__ T buf[Q * N];
    const int L = a.levels, at = (int)threadIdx.x;
    const int tile = (int)(blockIdx.x & 7) * a.chunk + (int)(blockIdx.x >> 3);
    if (tile >= a.tiles) return;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
    const int hy = at / W, hx = at - hy * W;
    const int ux = tx * kAdjTile - H + hx, uy = ty * kAdjTile - H + hy;
    const int x = wrap(ux, p.nx), y = wrap(uy, p.ny);
    const int xm = x == 0 ? p.nx - 1 : x - 1, xp = x == p.nx - 1 ? 0 : x + 1;
    const int ym = y == 0 ? p.ny - 1 : y - 1, yp = y == p.ny - 1 ? 0 : y + 1;
    const int ring = at < N ? max(0, max(max(H - hx, hx - (H + kAdjTile - 1)),
                                         max(H - hy, hy - (H + kAdjTile - 1)))) : kAdjLevels;
    const bool mine = ring == 0 && ux < p.nx && uy < p.ny;
    const long long n = (long long)x + (long long)p.nx * y;
    T f[Q], mu[Q], out[Q];
    auto load_state = [&](int l) {
        const S *src = static_cast<const S *>(a.state[l - 1]);
        const bool own = l == L && a.direct;
        const int sxm = own ? x : xm, sxp = own ? x : xp, sym = own ? y : ym, syp = own ? y : yp;
        LBM_ADJ_EACH([&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
            const int sx = cx == 0 ? x : (cx > 0 ? sxm : sxp), sy = cy == 0 ? y : (cy > 0 ? sym : syp);
            f[i] = ST::decode(src[p.plane * i + ((long long)sx + (long long)p.nx * sy)], i, p);
        });
    };
    double g0 = 0.0, g1 = 0.0;
    if (mine) {
        g0 = gtau[n];
        if constexpr (COLL == 1) g1 = gtau[p.plane + n];
    }
    if (ring <= L - 1) {
        load_state(1);
        LBM_ADJ_EACH([&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            constexpr int cx = QT<QID>::cx(i), cy = QT<QID>::cy(i);
            const int sx = cx == 0 ? x : (cx > 0 ? xp : xm), sy = cy == 0 ? y : (cy > 0 ? yp : ym);
            mu[i] = lam_next[p.plane * i + ((long long)sx + (long long)p.nx * sy)];
        });
    }
    for (int l = 1;; ++l) {
        if (ring <= L - l) {
            T gs, ga;
            adj_node<QID, ST, COLL>(f, mu, p, out, gs, ga);
            if (mine) adj_tau<COLL>(gs, ga, p, g0, g1);
        }
        if (l == L) break;
        if (ring <= L - l) {
            LBM_ADJ_EACH([&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                buf[N * i + at] = out[i];
            });
        }
        if (ring <= L - l - 1) load_state(l + 1);
        __syncthreads();
        if (ring <= L - l - 1) {
            LBM_ADJ_EACH([&](auto Ic) {
                constexpr int i = decltype(Ic)::value;
                mu[i] = buf[N * i + at + QT<QID>::cx(i) + W * QT<QID>::cy(i)];
            });
        }
        __syncthreads();
    }
    if (mine) {
        LBM_ADJ_EACH([&](auto Ic) {
            constexpr int i = decltype(Ic)::value;
            lam[p.plane * i + n] = out[i];
        });
        gtau[n] = g0;
        if constexpr (COLL == 1) gtau[p.plane + n] = g1;
    }
}

// lambda_T = dL/dS_T and the per-node loss 1/2 |u - u_target|^2
template <int QID, class ST, bool DIRECT>
__global__ void __launch_bounds__(256)
k_adj_seed(const typename ST::store_t *__restrict__ src, const double *__restrict__ ut,
           typename ST::T *__restrict__ lam, double *__restrict__ lossn, double *__restrict__ uT,
           const StepParams<typename ST::T> p) {
    using T = typename ST::T;
    constexpr int Q = QT<QID>::Q;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= p.nx) return;
    const long long n = (long long)x + (long long)p.nx * y;
    T f[Q];
    adj_state<QID, ST, DIRECT>(src, p, x, y, n, f);
    T drho, rho, ux, uy;
    adj_moments<QID, ST>(f, p, drho, rho, ux, uy);
    const double dx = static_cast<double>(ux) - ut[n];
    const double dy = static_cast<double>(uy) - ut[p.plane + n];
    lossn[n] = 0.5 * (dx * dx + dy * dy);
    if (uT) {
        uT[n] = static_cast<double>(ux);
        uT[p.plane + n] = static_cast<double>(uy);
    }
    const double ir = 1.0 / static_cast<double>(rho);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int j = decltype(Ic)::value;
        const double cx = QT<QID>::cx(j), cy = QT<QID>::cy(j);
        lam[p.plane * j + n] = static_cast<T>(
            (dx * (cx - static_cast<double>(ux)) + dy * (cy - static_cast<double>(uy))) * ir);
    });
}

// S_0 = feq(rho0, u0) (the reference's equilibrium initial condition,
// initial_conditions.jl:7-22, at uniform density)
template <int QID, class ST>
__global__ void __launch_bounds__(256)
k_adj_init(const double *__restrict__ u0, typename ST::store_t *__restrict__ S,
           const StepParams<typename ST::T> p) {
    using T = typename ST::T;
    constexpr int Q = QT<QID>::Q;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= p.nx) return;
    const long long n = (long long)x + (long long)p.nx * y;
    const T ux = static_cast<T>(u0[n]), uy = static_cast<T>(u0[p.plane + n]);
    const T usq = ux * ux + uy * uy;
    T f[Q];
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        if constexpr (ST::kShift) f[i] = feq_dev_i<QID, i, T>(T(0), p.rho0, ux, uy, usq, p);
        else f[i] = feq_i<QID, i, T>(p.rho0, ux, uy, usq, p);
    });
    store_local<QID, ST>(S, p, n, f, LBM_SEQ);
}

// dL/du0 = sum_i lambda_0,i dfeq_i(rho0, u0)/du0
template <int QID, class ST>
__global__ void __launch_bounds__(256)
k_adj_grad_u0(const double *__restrict__ u0, const typename ST::T *__restrict__ lam0,
              double *__restrict__ grad, const StepParams<typename ST::T> p) {
    using T = typename ST::T;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= p.nx) return;
    const long long n = (long long)x + (long long)p.nx * y;
    const T ux = static_cast<T>(u0[n]), uy = static_cast<T>(u0[p.plane + n]);
    const T usq = ux * ux + uy * uy;
    T gxs = T(0), gys = T(0);
    LBM_ADJ_EACH([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        T gx, gy;
        dfeq_du<QID, i, T>(p.rho0, ux, uy, usq, p, gx, gy);
        const T l = lam0[p.plane * i + n];
        gxs = gxs + l * gx;
        gys = gys + l * gy;
    });
    grad[n] = static_cast<double>(gxs);
    grad[p.plane + n] = static_cast<double>(gys);
}

template <int QID, class ST>
int launch_adjoint(const AdjLaunch &L, const StepParams<typename ST::T> &p, hipStream_t s) {
    using S = typename ST::store_t;
    using T = typename ST::T;
    const int bx = default_block(p.nx);
    const dim3 grid = node_grid(p.nx, p.ny, bx), block(bx, 1, 1);
    const S *st = static_cast<const S *>(L.state);
    const T *li = static_cast<const T *>(L.lam_in);
    T *lo = static_cast<T *>(L.lam_out);
    switch (L.what) {
    case 0:
        k_adj_init<QID, ST><<<grid, block, 0, s>>>(L.u, static_cast<S *>(L.pops), p);
        break;
    case 1:
        if (L.direct) k_adj_seed<QID, ST, true><<<grid, block, 0, s>>>(st, L.u, lo, L.out, L.aux, p);
        else k_adj_seed<QID, ST, false><<<grid, block, 0, s>>>(st, L.u, lo, L.out, L.aux, p);
        break;
    case 2:
        if (L.coll == 0) {
            if (L.direct) k_adj_step<QID, ST, 0, true><<<grid, block, 0, s>>>(li, st, lo, L.out, p);
            else k_adj_step<QID, ST, 0, false><<<grid, block, 0, s>>>(li, st, lo, L.out, p);
        } else if (L.coll == 1) {
            if (L.direct) k_adj_step<QID, ST, 1, true><<<grid, block, 0, s>>>(li, st, lo, L.out, p);
            else k_adj_step<QID, ST, 1, false><<<grid, block, 0, s>>>(li, st, lo, L.out, p);
        } else {
            return -2;
        }
        break;
    case 4:
        if constexpr (QT<QID>::MAXC == 1) {
            if (L.levels < 1 || L.levels > kAdjLevels) return -5;
            AdjLevels a;
            for (int l = 0; l < kAdjLevels; ++l) a.state[l] = L.states[l];
            a.levels = L.levels;
            a.direct = L.direct;
            a.tiles_x = (p.nx + kAdjTile - 1) / kAdjTile;
            a.tiles = a.tiles_x * ((p.ny + kAdjTile - 1) / kAdjTile);
            a.chunk = (a.tiles + 7) / 8;
            const unsigned tiles = 8u * (unsigned)a.chunk;
            if (L.coll == 0) k_adj_tile<QID, ST, 0><<<tiles, kAdjThreads, 0, s>>>(li, lo, L.out, p, a);
            else if constexpr (!ST::kShift)
                k_adj_tile<QID, ST, 1><<<tiles, kAdjThreads, 0, s>>>(li, lo, L.out, p, a);
            else return -2;
            break;
        } else {
            return -3;
        }
    case 3:
        k_adj_grad_u0<QID, ST><<<grid, block, 0, s>>>(L.u, li, L.out, p);
        break;
    default:
        return -3;
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

#define LBM_DEFINE_ADJOINT(TAG, ST)                                                          \
    int run_adjoint_##TAG(const AdjLaunch &L, const StepParams<typename ST::T> &p,           \
                          hipStream_t s) {                                                   \
        switch (L.qid) {                                                                     \
        case 4: return launch_adjoint<4, ST>(L, p, s);                                       \
        case 5: return launch_adjoint<5, ST>(L, p, s);                                       \
        case 9: return launch_adjoint<9, ST>(L, p, s);                                       \
        case 13: return launch_adjoint<13, ST>(L, p, s);                                     \
        case 17: return launch_adjoint<17, ST>(L, p, s);                                     \
        case 21: return launch_adjoint<21, ST>(L, p, s);                                     \
        case 37: return launch_adjoint<37, ST>(L, p, s);                                     \
        default: return -1;                                                                  \
        }                                                                                    \
    }

}  // namespace lbm
