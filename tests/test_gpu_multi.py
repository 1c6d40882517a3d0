"""Runs that advance several steps per pass (lbm_multi.h) against the oracle.

A run without a launch shape picks its kernel by the number of nodes: 8 x 8
tiles, register blocks of 64 x 16, 64 x 32 and 64 x 24 (FP32 64 x 32) nodes,
marching waves.  The shapes below sit at every kernel's edges: lattices
narrower or lower than one tile (the halo wraps several times), the narrowest
and lowest ones that the wide kernels take (32 columns, 12 rows) and those
just below, widths and heights that leave remainders, step counts that need
every pass size."""
import numpy as np
import pytest

from lbm_cases import bc_dicts, force_for, random_populations, to_lbmhip

pytestmark = pytest.mark.gpu

# (nx, ny): by kernel, smallest to largest
TILE = [(1, 1), (2, 3), (3, 40), (9, 8), (64, 64), (200, 199)]
# (the steps per pass of a block kernel differ by shape)
BLOCK16 = [(257, 160), (32, 2500), (9001, 12), (31, 2501), (9001, 11), (300, 300), (340, 340),
           (380, 380)]
BLOCK32 = [(513, 300), (55, 2500), (460, 460), (560, 560), (600, 600)]
WIDE = [(1021, 517), (57, 8001), (700, 700), (760, 760), (2049, 1000), (33, 61001), (170001, 12)]
MARCH = [(2049, 1500), (47, 65001), (250001, 12), (1200001, 3)]
SHAPES = TILE + BLOCK16 + BLOCK32 + WIDE + MARCH


def _L():
    import lbmhip
    return lbmhip


def _populations(qid, nx, ny, seed, noise=2e-3):
    """A random field of at most 61 x 53 nodes, repeated over the lattice."""
    f = random_populations(qid, min(nx, 61), min(ny, 53), seed=seed, noise=noise)
    reps = (-(-nx // f.shape[0]), -(-ny // f.shape[1]), 1)
    return np.asfortranarray(np.tile(f, reps)[:nx, :ny])


def _model(qid, coll, F):
    L = _L()
    q = L.Quadratures[f"D2Q{qid}"]()
    if coll == 0:
        return q, L.SRT(0.8, F), [0.8]
    if coll == 1:
        return q, L.TRT.fields(0.7, 1.3, F), [0.7, 1.3]
    return q, L.MRT(q, [0.9, 0.75], force=F), [0.9, 0.75]


def _oracle(oracle_lib, qid, f0, coll, taus, steps, F, bcs):
    S, C = f0.copy(order="F"), f0.copy(order="F")
    oracle_lib.set_threads(16)
    try:
        oracle_lib.simulate(qid, S, C, coll, taus, steps, force=F, bcs=bcs)
    finally:
        oracle_lib.set_threads(1)
    return S, C


def _check_f64(oracle_lib, qid, coll, nx, ny, bcname, force, steps):
    f0 = _populations(qid, nx, ny, seed=qid + 3 * coll)
    F = force_for(force, nx, ny)
    q, cm, taus = _model(qid, coll, F)
    bcs = bc_dicts(bcname, nx, ny)
    model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs))
    print(f"multi D2Q{qid} coll {coll} {nx}x{ny} {bcname} {force} {steps} steps", flush=True)
    _L().simulate(model, range(steps))
    S, C = _oracle(oracle_lib, qid, f0, coll, taus, steps, F, bcs)
    assert np.array_equal(model.f_stream.to_numpy(), S), (nx, ny, steps)
    assert np.array_equal(model.f_collision.to_numpy(), C), (nx, ny, steps)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("coll,bcname,force,steps", [
    (0, "periodic", "none", 11), (1, "cavity", "field", 13), (2, "partial", "const", 9)])
def test_f64_bit_exact(oracle_lib, shape, coll, bcname, force, steps):
    _check_f64(oracle_lib, 9, coll, *shape, bcname, force, steps)


@pytest.mark.parametrize("shape", [(70, 33), (257, 160), (1021, 517)])
@pytest.mark.parametrize("steps", range(2, 9))
def test_f64_every_pass_size(oracle_lib, shape, steps):
    _check_f64(oracle_lib, 9, 1, *shape, "couette", "const", steps)


@pytest.mark.parametrize("steps", [2, 3, 4, 6, 7])
def test_f64_march_pass_sizes(oracle_lib, steps):
    _check_f64(oracle_lib, 9, 1, 2049, 1500, "couette", "const", steps)


@pytest.mark.parametrize("qid", [4, 5])
@pytest.mark.parametrize("coll", [0, 1, 2])
@pytest.mark.parametrize("shape", [(19, 40), (257, 160), (513, 300), (700, 650), (2049, 1500)])
def test_f64_other_one_speed_sets(oracle_lib, qid, coll, shape):
    _check_f64(oracle_lib, qid, coll, *shape, "cavity", "const", 9)


@pytest.mark.parametrize("coll", [0, 1])
@pytest.mark.parametrize("shape", [(3, 40), (64, 64), (257, 160), (513, 300), (1021, 517),
                                   (2050, 1000), (33, 61001), (300, 300), (340, 340), (380, 380),
                                   (460, 460), (560, 560), (4097, 2500), (161, 65001)])
@pytest.mark.parametrize("bcname,force", [("periodic", "none"), ("cavity", "field")])
def test_f32_tracks_oracle(oracle_lib, coll, shape, bcname, force):
    """FP32 on shifted populations |g| = |f - w| <= G: a step's rounding errors
    are below 16 half-ulps of G per population (the pair sums, the
    equilibrium's five operations, the relaxation), and the collision with
    tau > 1/2 carries a deviation on with a factor of at most 1 in the summed
    norm, so after n steps |error| <= 16 n 2^-24 G with room for the initial
    rounding."""
    nx, ny = shape
    steps = 13
    f0 = _populations(9, nx, ny, seed=5, noise=1e-4)
    F = force_for(force, nx, ny)
    q, cm, taus = _model(9, coll, F)
    bcs = bc_dicts(bcname, nx, ny)
    m = _L().LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage="f32")
    _L().simulate(m, range(steps))
    S, C = _oracle(oracle_lib, 9, f0, coll, taus, steps, F, bcs)
    w = np.asarray(q.weights)
    G = max(np.abs(S - w).max(), np.abs(C - w).max(), np.abs(f0 - w).max())
    tol = 16 * (steps + 1) * 2.0 ** -24 * G
    assert np.abs(m.f_stream.to_numpy() - S).max() <= tol
    assert np.abs(m.f_collision.to_numpy() - C).max() <= tol


@pytest.mark.parametrize("storage", ["f16neq", "bf16neq"])
@pytest.mark.parametrize("qid", [4, 5, 9])
@pytest.mark.parametrize("coll", [0, 1])
@pytest.mark.parametrize("shape", [(1022, 800), (112, 7200), (64, 12600), (66700, 12)])
@pytest.mark.parametrize("bcname,force,steps", [("periodic", "none", 2), ("cavity", "field", 9),
                                                ("couette", "const", 11)])
def test_neq_error_no_larger_than_single_steps(oracle_lib, storage, qid, coll, shape, bcname,
                                               force, steps):
    """The 16-bit storages round once per pass instead of once per step: the
    populations' error against the oracle's FP64 run is at most that of the
    single-step kernels (which the per-launch timing entry point keeps), with
    a tenth for the scatter of roundings."""
    L = _L()
    nx, ny = shape
    f0 = _populations(qid, nx, ny, seed=7, noise=1e-4)
    F = force_for(force, nx, ny)
    q, cm, taus = _model(qid, coll, F)
    bcs = bc_dicts(bcname, nx, ny)
    many = L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage=storage)
    L.simulate(many, range(steps))
    one = L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage=storage)
    L.simulate_launch_times(one, steps)
    S, C = _oracle(oracle_lib, qid, f0, coll, taus, steps, F, bcs)
    for a, b, ref in ((many.f_stream, one.f_stream, S), (many.f_collision, one.f_collision, C)):
        ea, eb = (np.linalg.norm(x.to_numpy() - ref) for x in (a, b))
        assert ea <= 1.1 * eb, (ea, eb)


# a batch: widths and heights at one and two blocks' outputs (56 x 16 FP64,
# 54 x 22 FP32) and beside them, narrower and lower than a block's halo, long
# rows; big enough on average for the several-step passes
BATCH = [(56, 16), (57, 17), (54, 22), (300, 129), (113, 45), (129, 200), (7, 90), (200, 5),
         (256, 256), (1, 64), (64, 1), (333, 77)]


def _batch(storage, trt, noise):
    rng = np.random.default_rng(3)
    ts = rng.uniform(0.55, 1.4, len(BATCH))
    ta = 0.5 + 0.25 / (ts - 0.5) if trt else None
    L = _L()
    b = L.LatticeBatch(L.D2Q9(), BATCH, ts, ta, storage=storage)
    f0 = [_populations(9, nx, ny, seed=k, noise=noise) for k, (nx, ny) in enumerate(BATCH)]
    for k, f in enumerate(f0):
        b.upload(k, f)
        if storage == "f64":
            assert np.array_equal(b.download(k, "f_collision"), f)
    return b, f0, [[ts[k], ta[k]] if trt else [ts[k]] for k in range(len(BATCH))]


@pytest.mark.parametrize("trt", [False, True])
@pytest.mark.parametrize("calls", [(1, 2), (3, 1), (4,), (5,), (6, 7), (23,)])
def test_batch_f64_bit_exact(oracle_lib, trt, calls):
    b, f0, taus = _batch("f64", trt, 2e-3)
    print(f"batch f64 trt {trt} {calls}", flush=True)
    for n in calls:
        b.simulate(n)
    b.set_launch(64, 0)  # the single-step kernel goes on from the same state
    b.simulate(2)
    b.set_launch(0, 0)
    b.simulate(2)
    for k, f in enumerate(f0):
        S, C = _oracle(oracle_lib, 9, f, int(trt), taus[k], sum(calls) + 4, None, [])
        assert np.array_equal(b.download(k, "f_stream"), S), BATCH[k]
        assert np.array_equal(b.download(k, "f_collision"), C), BATCH[k]


@pytest.mark.parametrize("trt", [False, True])
@pytest.mark.parametrize("steps", [2, 6, 13])
def test_batch_f32_tracks_oracle(oracle_lib, trt, steps):
    """the bound of test_f32_tracks_oracle, lattice by lattice"""
    b, f0, taus = _batch("f32", trt, 1e-4)
    b.simulate(steps)
    w = np.asarray(_L().D2Q9().weights)
    for k, f in enumerate(f0):
        S, C = _oracle(oracle_lib, 9, f, int(trt), taus[k], steps, None, [])
        G = max(np.abs(S - w).max(), np.abs(C - w).max(), np.abs(f - w).max())
        tol = 16 * (steps + 1) * 2.0 ** -24 * G
        assert np.abs(b.download(k, "f_stream") - S).max() <= tol, BATCH[k]
        assert np.abs(b.download(k, "f_collision") - C).max() <= tol, BATCH[k]


# the iterative initialization: up to 420 tiles (168 x 160) several steps a
# launch, beyond them and on the other stencils one
MEI = [(9, 5, 7), (9, 33, 20), (9, 168, 160), (9, 169, 160), (4, 24, 31), (5, 24, 31),
       (13, 40, 17), (17, 70, 9), (37, 20, 33)]


def _mei_run(qid, u, bcs, eps, max_steps):
    import ctypes
    L = _L()
    from lbmhip import _lib
    from lbmhip.operators import native_model
    q = L.Quadratures[f"D2Q{qid}"]()
    nx, ny = u.shape[:2]
    fs, fc = L.HipLattice(q, nx, ny), L.HipLattice(q, nx, ny)
    m = native_model(q).configure(L.IterativeInitializationCollisionModel(0.8, u), fs, bcs)
    steps = ctypes.c_int64()
    _lib.check(_lib.lib().lbm_mei_initialize(m.handle, fs.handle, fc.handle, eps, max_steps,
                                             ctypes.byref(steps)), "lbm_mei_initialize")
    return fs.to_numpy(), fc.to_numpy(), steps.value


@pytest.mark.parametrize("qid,nx,ny", MEI)
@pytest.mark.parametrize("bcname", ["periodic", "couette"])
@pytest.mark.parametrize("eps,max_steps", [
    (0.0, 1), (0.0, 2), (0.0, 9), (0.0, 10), (0.0, 41), (2.0, 30),
    (5e-3, 200), (3e-3, 200), (1e-3, 200), (5e-4, 200), (1e-4, 200), (1e-6, 200)])
def test_mei_initialize_bit_exact(oracle_lib, qid, nx, ny, bcname, eps, max_steps):
    """steps run, f_stream and f_collision, with stops inside and at the ends
    of passes"""
    x, y = np.meshgrid(np.arange(nx) * 2 * np.pi / nx, np.arange(ny) * 2 * np.pi / ny,
                       indexing="ij")
    u = np.asfortranarray(np.stack([0.03 * np.cos(x) * np.sin(y), 0.02 * np.sin(x + y)], axis=-1))
    bcd = bc_dicts(bcname, nx, ny)
    print(f"mei D2Q{qid} {nx}x{ny} {bcname} eps {eps} {max_steps}", flush=True)
    S, C, n = oracle_lib.mei_initialize(qid, u, 0.8, eps, max_steps, bcd)
    s, c, steps = _mei_run(qid, u, to_lbmhip(bcd), eps, max_steps)
    assert steps == n
    assert np.array_equal(s, S)
    assert np.array_equal(c, C)


# the reverse pass: 16 x 16 tiles of up to four steps, forward and recomputed
# segments by every several-step kernel and, at 31 x 2501, single steps
ADJOINT = [(1, 1), (2, 3), (16, 16), (17, 33), (130, 47), (257, 160), (340, 340), (513, 300),
           (700, 650), (31, 2501), (2049, 1500)]


def _adjoint(qid, coll, shape, T, K, storage, u0, ut):
    L = _L()
    cm = L.SRT(0.8) if coll == 0 else L.TRT.fields(0.75, 1.2)
    prob = L.AdjointProblem(L.Quadratures[f"D2Q{qid}"](), cm, shape, T, storage=storage,
                            checkpoint_every=K)
    r = prob.gradient(u0, ut)
    prob.close()
    return r


@pytest.mark.parametrize("qid,shape", [(9, s) for s in ADJOINT] +
                         [(4, (130, 47)), (5, (130, 47)), (5, (257, 160))])
@pytest.mark.parametrize("coll", [0, 1])
@pytest.mark.parametrize("T", [2, 11, 13])
def test_adjoint_passes(qid, shape, coll, T):
    """FP64: single steps (a checkpoint at each step) and passes give the same
    bits.  FP32 against FP64: a step rounds each of its terms a few times, 64
    half-ulps in the summed norm with the forward run's share, so after T
    steps the relative difference is below 64 (T + 1) 2^-24."""
    rng = np.random.default_rng(T)
    u0, ut = (0.03 * rng.standard_normal((*shape, 2)) for _ in (0, 1))
    print(f"adjoint D2Q{qid} {shape} coll {coll} T {T}", flush=True)
    ref = _adjoint(qid, coll, shape, T, 1, "f64", u0, ut)
    for K in (0, 3, T):
        r = _adjoint(qid, coll, shape, T, K, "f64", u0, ut)
        assert r["loss"] == ref["loss"], K
        assert np.array_equal(r["grad_u0"], ref["grad_u0"]), K
        assert np.array_equal(r["grad_tau"], ref["grad_tau"]), K
    r = _adjoint(qid, coll, shape, T, T, "f32", u0, ut)
    tol = 64 * (T + 1) * 2.0 ** -24
    assert np.linalg.norm(r["grad_u0"] - ref["grad_u0"]) <= tol * np.linalg.norm(ref["grad_u0"])
    assert abs(r["loss"] - ref["loss"]) <= tol * ref["loss"]


def _corner_changes(oracle_lib, qid, u, steps, bcs):
    """|rho_t - rho_(t-1)| at node (nx, ny), t = 1 .. steps, rho_0 = 0"""
    rho, out = 0.0, []
    for t in range(1, steps + 1):
        S, _, _ = oracle_lib.mei_initialize(qid, u, 0.8, 0.0, t, bcs)
        r = S[-1, -1, 0] + S[-1, -1, 1]
        for i in range(2, S.shape[2]):
            r = r + S[-1, -1, i]
        out.append(abs(r - rho))
        rho = r
    return out


@pytest.mark.parametrize("qid,nx,ny", [(9, 33, 20), (9, 5, 7), (9, 168, 160), (9, 169, 160),
                                       (5, 24, 31), (13, 40, 17)])
@pytest.mark.parametrize("bcname", ["periodic", "couette"])
def test_mei_stop_at_every_step_that_can_hold_it(oracle_lib, qid, nx, ny, bcname):
    """The recording launch is run by all its threads to its end (it has
    barriers), the ones after it by none: wherever in a launch the stop falls,
    steps, f_stream and f_collision are the oracle's."""
    x, y = np.meshgrid(np.arange(nx) * 2 * np.pi / nx, np.arange(ny) * 2 * np.pi / ny,
                       indexing="ij")
    u = np.asfortranarray(np.stack([0.03 * np.cos(x) * np.sin(y), 0.02 * np.sin(x + y)], axis=-1))
    bcd = bc_dicts(bcname, nx, ny)
    d = _corner_changes(oracle_lib, qid, u, 26, bcd)
    low, at = d[0], [1]
    for t in range(2, len(d) + 1):
        if d[t - 1] < low:
            at.append(t)
            low = d[t - 1]
    print(f"mei stops D2Q{qid} {nx}x{ny} {bcname}: {at}", flush=True)
    assert len(at) > 1
    for t in at:
        eps = 1.5 * d[0] if t == 1 else 0.5 * (min(d[:t - 1]) + d[t - 1])
        S, C, n = oracle_lib.mei_initialize(qid, u, 0.8, eps, 200, bcd)
        assert n == t
        s, c, steps = _mei_run(qid, u, to_lbmhip(bcd), eps, 200)
        assert steps == t
        assert np.array_equal(s, S)
        assert np.array_equal(c, C)


@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_batch_transfers_from_several_threads(storage):
    """Threads that move different lattices of one batch at a time share its
    transfer buffer, which grows with the lattice: every thread gets back what
    it put in."""
    from concurrent.futures import ThreadPoolExecutor
    L = _L()
    sizes = [(8 + 37 * k, 5 + 23 * k) for k in range(12)]
    b = L.LatticeBatch(L.D2Q9(), sizes, [0.8] * len(sizes), None, storage=storage)
    f = [_populations(9, nx, ny, seed=k) for k, (nx, ny) in enumerate(sizes)]
    if storage == "f32":  # values that FP32 holds, as deviations from the weights too
        w = np.asarray(L.D2Q9().weights)
        dev = [np.round((x - w) * 2.0 ** 20) * 2.0 ** -20 for x in f]
        f = [np.asfortranarray(w.astype(np.float32).astype(float) + d) for d in dev]

    def move(k):
        for _ in range(20):
            b.upload(k, f[k])
            for role in ("f_stream", "f_collision"):
                np.testing.assert_allclose(b.download(k, role), f[k], rtol=0,
                                           atol=0 if storage == "f64" else 2.0 ** -26)

    with ThreadPoolExecutor(4) as pool:
        list(pool.map(move, range(len(sizes))))


def _ranged_walls(nx, ny):
    """East and west walls whose ranges begin and end at rows all over the
    lattice, one row long too, a later condition over an earlier one."""
    return [dict(kind=0, direction=1, xs=(1, nx), ys=(min(7, ny), max(min(7, ny), ny // 3))),
            dict(kind=0, direction=1, xs=(1, nx), ys=(ny // 2, ny // 2)),
            dict(kind=0, direction=3, xs=(1, nx), ys=(ny // 2, ny)),
            dict(kind=0, direction=3, xs=(1, nx), ys=(1, 1)),
            dict(kind=1, direction=0, xs=(1, nx), ys=(1, ny), u=(0.05, 0.0), rho=1.0),
            dict(kind=0, direction=0, xs=(nx // 2, nx), ys=(2, ny)),
            dict(kind=0, direction=2, xs=(2, nx // 3), ys=(1, ny))]


@pytest.mark.parametrize("shape", [(2049, 1500), (47, 65001), (250001, 12)])
@pytest.mark.parametrize("coll,steps", [(0, 5), (1, 13)])
def test_march_ranged_walls_f64_bit_exact(oracle_lib, shape, coll, steps):
    nx, ny = shape
    f0 = _populations(9, nx, ny, seed=17)
    q, cm, taus = _model(9, coll, None)
    bcs = _ranged_walls(nx, ny)
    model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs))
    print(f"march ranges {nx}x{ny} coll {coll} {steps} steps", flush=True)
    _L().simulate(model, range(steps))
    S, C = _oracle(oracle_lib, 9, f0, coll, taus, steps, None, bcs)
    assert np.array_equal(model.f_stream.to_numpy(), S)
    assert np.array_equal(model.f_collision.to_numpy(), C)


@pytest.mark.parametrize("storage", ["f16neq", "bf16neq"])
@pytest.mark.parametrize("qid", [4, 9])
@pytest.mark.parametrize("shape,bcname", [((1500, 1204), "ranged"), ((1500, 1204), "cavity"),
                                          ((1202, 1000), "couette"), ((64, 19001), "ranged"),
                                          ((150002, 12), "partial")])
def test_march_walls_neq_error_no_larger_than_single_steps(oracle_lib, storage, qid, shape, bcname):
    """as test_neq_error_no_larger_than_single_steps, on lattices that their
    walls leave to the several-step kernel"""
    L = _L()
    nx, ny = shape
    f0 = _populations(qid, nx, ny, seed=7, noise=1e-4)
    q, cm, taus = _model(qid, 1, None)
    bcs = _ranged_walls(nx, ny) if bcname == "ranged" else bc_dicts(bcname, nx, ny)
    many = L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage=storage)
    L.simulate(many, range(9))
    one = L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage=storage)
    L.simulate_launch_times(one, 9)
    S, C = _oracle(oracle_lib, qid, f0, 1, taus, 9, None, bcs)
    for a, b, ref in ((many.f_stream, one.f_stream, S), (many.f_collision, one.f_collision, C)):
        ea, eb = (np.linalg.norm(x.to_numpy() - ref) for x in (a, b))
        assert ea <= 1.1 * eb, (ea, eb)


@pytest.mark.parametrize("shape", [(64, 8000), (6400, 64), (4096, 2048), (128, 8000)])
@pytest.mark.parametrize("coll,bcname", [(1, "periodic"), (2, "cavity")])
def test_two_steps_on_whole_tiles_f64_bit_exact(oracle_lib, shape, coll, bcname):
    """a run of two steps keeps the single-step kernels' one-pass start on
    large lattices and on narrow or low ones"""
    _check_f64(oracle_lib, 9, coll, *shape, bcname, "const", 2)


# densities at the ends of div2's range (2^-510 .. 2^510) and beyond it, zero and
# negative ones, momenta far below their density
SCALES = [1.0, 2.0 ** -400, 2.0 ** -509, 2.0 ** -511, 2.0 ** -520, 2.0 ** -1000, 2.0 ** 400,
          2.0 ** 509, 2.0 ** 511, 2.0 ** 700, 0.0, -1.0, -(2.0 ** -515), -(2.0 ** 300)]


@pytest.mark.parametrize("qid,shape", [(9, (100, 90)), (9, (300, 250)), (9, (2049, 1500)),
                                       (17, (600, 500))])
@pytest.mark.parametrize("coll", [0, 1, 2])
@pytest.mark.parametrize("whole", [True, False])
@pytest.mark.parametrize("force", ["none", "const"])
def test_f64_extreme_densities_bit_exact(oracle_lib, qid, shape, coll, whole, force):
    """The shared reciprocal of the several-step kernels gives the plain
    divisions' populations: whole lattices of one scale, and nodes of all scales
    side by side."""
    if qid == 17 and coll == 2:
        pytest.skip("MRT on D2Q17 runs single steps")
    nx, ny = shape
    q, cm, taus = _model(qid, coll, force_for(force, nx, ny))
    base = _populations(qid, nx, ny, seed=4)
    scales = SCALES if whole and nx < 600 else [None]
    for s in scales:
        if s is not None:
            f0 = base * s
        else:
            k = np.random.default_rng(1).integers(0, len(SCALES), (nx, ny))
            f0 = np.asfortranarray(base * np.asarray(SCALES)[k][:, :, None])
            f0[::7, ::5, :] = 0.0  # momentum 2^-960 .. 2^-1074 of a density of one
            f0[::7, ::5, 0] = 1.0
            f0[::7, ::5, 2] = 2.0 ** -np.random.default_rng(2).integers(950, 1074, f0[::7, ::5, 2].shape)
        model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm)
        print(f"extreme D2Q{qid} {nx}x{ny} coll {coll} scale {s}", flush=True)
        _L().simulate(model, range(3))
        S, C = _oracle(oracle_lib, qid, f0, coll, taus, 3, force_for(force, nx, ny), [])
        assert np.array_equal(model.f_stream.to_numpy(), S, equal_nan=True), s
        assert np.array_equal(model.f_collision.to_numpy(), C, equal_nan=True), s


@pytest.mark.parametrize("qid,shape", [(9, (100, 90)), (9, (300, 250)), (9, (2049, 1500)),
                                       (17, (600, 500))])
@pytest.mark.parametrize("coll", [0, 1])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, pytest.param(1.7e308, marks=pytest.mark.xfail(
    reason="the pair form carries the halves of the relaxation in its rates: a difference of "
           "pair sums beyond 2^1023 overflows where halves of them would not"))])
def test_f64_non_finite_populations(oracle_lib, qid, shape, coll, value):
    """NaN and infinities spread as in the oracle, and no further"""
    nx, ny = shape
    q, cm, taus = _model(qid, coll, None)
    f0 = _populations(qid, nx, ny, seed=4)
    for i in range(q.Q):
        f0[(11 * i + 3) % nx, (17 * i + 2) % ny, i] = value
    f0[nx // 2, ny // 2, :] = value
    model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm)
    print(f"non-finite D2Q{qid} {nx}x{ny} coll {coll} {value}", flush=True)
    _L().simulate(model, range(4))
    with np.errstate(all="ignore"):
        S, C = _oracle(oracle_lib, qid, f0, coll, taus, 4, None, [])
    assert np.isnan(S).any() or np.isinf(S).any()
    assert np.array_equal(model.f_stream.to_numpy(), S, equal_nan=True)
    assert np.array_equal(model.f_collision.to_numpy(), C, equal_nan=True)


def _vortices(nx, ny, seed):
    rng = np.random.default_rng(seed)
    x, y = np.meshgrid(np.arange(nx) * 2 * np.pi / nx, np.arange(ny) * 2 * np.pi / ny,
                       indexing="ij")
    ux, uy = (sum(0.01 * rng.normal() * np.sin(k * c + rng.uniform(0, 6)) for k in (1, 2, 3))
              for c in (y, x))
    return 1 + 0.01 * np.sin(x + y), ux, uy


@pytest.mark.parametrize("qid", [4, 5, 9])
@pytest.mark.parametrize("shape", [(100, 90), (300, 250), (1021, 517), (4099, 2500)])
@pytest.mark.parametrize("coll,tau", [(0, 0.6), (0, 0.678), (0, 0.728), (0, 0.87), (0, 0.949),
                                      (0, 0.969), (1, 0.6), (1, 0.668), (1, 0.8)])
def test_f32_drift_no_larger_than_single_steps(qid, shape, coll, tau):
    """FP32 over 200 steps: what a step's rounding adds up to (the drift of the
    momentum, which depends on how a form rounds the weights and rates) is at
    most the single-step kernels', with a twentieth for scatter."""
    L = _L()
    q = L.Quadratures[f"D2Q{qid}"]()
    f0 = L.equilibrium_populations(q, *_vortices(*shape, seed=qid))
    cm = L.SRT(tau) if coll == 0 else L.trt_magic(tau)

    def run(storage, fn):
        m = L.LatticeBoltzmannModel.from_populations(q, f0, cm, storage=storage)
        fn(m)
        return m.f_stream.to_numpy()

    steps = 200 if shape[0] < 4000 else 40
    ref = run("f64", lambda m: L.simulate(m, range(steps)))
    many = np.linalg.norm(run("f32", lambda m: L.simulate(m, range(steps))) - ref)
    one = np.linalg.norm(run("f32", lambda m: L.simulate_launch_times(m, steps)) - ref)
    assert many <= 1.05 * one, (many / one)


@pytest.mark.parametrize("trt", [False, True])
def test_batch_f32_drift_no_larger_than_single_steps(trt):
    L = _L()
    sizes = [(100 + 10 * k, 90) for k in range(8)]
    taus = [0.6, 0.643, 0.678, 0.728, 0.8, 0.87, 0.949, 0.969]
    ta = [0.5 + 0.25 / (t - 0.5) for t in taus] if trt else None
    f0 = [L.equilibrium_populations(L.D2Q9(), *_vortices(*s, seed=k)) for k, s in enumerate(sizes)]

    def run(storage, shape):
        b = L.LatticeBatch(L.D2Q9(), sizes, taus, ta, storage=storage)
        for k, f in enumerate(f0):
            b.upload(k, f)
        b.set_launch(*shape)
        b.simulate(200)
        return [b.download(k) for k in range(len(sizes))]

    ref, many, one = run("f64", (0, 0)), run("f32", (0, 0)), run("f32", (128, 0))
    for k in range(len(sizes)):
        e = [np.linalg.norm(x[k] - ref[k]) for x in (many, one)]
        assert e[0] <= 1.05 * e[1], (taus[k], e)


@pytest.mark.parametrize("storage", ["f16neq", "bf16neq"])
@pytest.mark.parametrize("qid", [4, 5, 9])
@pytest.mark.parametrize("coll,tau", [(0, 0.6), (0, 0.643), (0, 0.8), (1, 0.6), (1, 0.678),
                                      (1, 0.728), (1, 0.9)])
def test_neq_drift_no_larger_than_single_steps(storage, qid, coll, tau):
    """the same for the 16-bit storages, 200 steps on 1000 x 900"""
    L = _L()
    q = L.Quadratures[f"D2Q{qid}"]()
    f0 = L.equilibrium_populations(q, *_vortices(1000, 900, seed=qid))
    cm = L.SRT(tau) if coll == 0 else L.trt_magic(tau)

    def run(st, fn):
        m = L.LatticeBoltzmannModel.from_populations(q, f0, cm, storage=st)
        fn(m)
        return m.f_stream.to_numpy()

    ref = run("f64", lambda m: L.simulate(m, range(200)))
    many = np.linalg.norm(run(storage, lambda m: L.simulate(m, range(200))) - ref)
    one = np.linalg.norm(run(storage, lambda m: L.simulate_launch_times(m, 200)) - ref)
    assert many <= 1.05 * one, (many / one)
