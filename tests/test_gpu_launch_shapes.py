"""Which kernels a run takes by its launch shape: a shape set by the caller
means one fused step per launch, the automatic setting several steps per pass.

FP32 TRT on D2Q9 tells the two apart: the several-step kernels round a step
differently.  ``simulate_launch_times`` runs one step per launch whatever the
shape."""
import numpy as np
import pytest

from lbm_cases import random_populations

pytestmark = pytest.mark.gpu


def _run(shape, launch, steps, times=False):
    import lbmhip as L
    f0 = random_populations(9, *shape, seed=3, noise=1e-2)
    m = L.LatticeBoltzmannModel.from_populations(L.D2Q9(), f0, L.TRT.fields(0.7, 1.3),
                                                 storage="f32")
    m.launch = launch
    if times:
        L.simulate_launch_times(m, steps)
    else:
        L.simulate(m, range(steps))
    return m.f_stream.to_numpy()


@pytest.mark.parametrize("shape", [(100, 90), (300, 250)])
def test_a_shape_set_to_the_automatic_numbers_runs_single_steps(shape):
    several = _run(shape, None, 9)
    for launch in ((256, 1, 1, 1), (256, 1, 1, 0), (0, 0, 0, 1), (128, 1, 1, -1)):
        single = _run(shape, launch, 9, times=True)
        assert not np.array_equal(single, several)
        assert np.array_equal(_run(shape, launch, 9), single), launch
    for launch in ((0, 0, 0, -1), (256, 1, 1, -1)):
        assert np.array_equal(_run(shape, launch, 9), several), launch


@pytest.mark.parametrize("shape", [(100, 90), (300, 250)])
def test_autotune_result_names_the_kernel_it_timed(shape):
    import lbmhip as L
    f0 = random_populations(9, *shape, seed=3, noise=1e-2)
    m = L.LatticeBoltzmannModel.from_populations(L.D2Q9(), f0, L.TRT.fields(0.7, 1.3),
                                                 storage="f32")
    best = L.autotune(m, trial_steps=20)
    L.simulate(m, range(9))
    several = _run(shape, None, 9)
    want = several if best["nontemporal"] < 0 else _run(shape, m.launch, 9, times=True)
    assert np.array_equal(m.f_stream.to_numpy(), want)
    # applied to another model
    assert np.array_equal(_run(shape, m.launch, 9), want)


SIZES = [(200, 100), (64, 64), (90, 70), (130, 48)]


def _batch():
    import lbmhip as L
    b = L.LatticeBatch(L.D2Q9(), SIZES, [0.7] * len(SIZES), [1.3] * len(SIZES), storage="f32")
    for k, shape in enumerate(SIZES):
        b.upload(k, random_populations(9, *shape, seed=k, noise=1e-2))
    return b


def _batch_run(launch):
    b = _batch()
    if launch is not None:
        b.set_launch(launch["block"], launch["grid"], launch["nodes_per_thread"])
    b.simulate(9)
    return b, [b.download(k) for k in range(len(b))]


def _equal(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_batch_shape_read_and_set_again_names_the_same_kernel():
    """the automatic setting, shapes with its numbers, and what the autotuner
    returns"""
    auto, several = _batch_run(None)
    tiles = sum(-(-(-(-nx // 32) * 32 * ny) // 128) for nx, ny in SIZES)
    shapes = [dict(block=128, grid=0, nodes_per_thread=1),
              dict(block=128, grid=tiles, nodes_per_thread=1)]
    single = _batch_run(shapes[0])[1]
    assert not _equal(single, several)
    assert _equal(_batch_run(auto.launch())[1], several)
    for s in shapes:
        b, got = _batch_run(s)
        assert b.launch() == s
        assert _equal(got, single), s
    b = _batch()
    best = b.autotune(5)
    shape = {k: best[k] for k in ("block", "grid", "nodes_per_thread")}
    b.simulate(9)
    assert b.launch() == shape
    got = [b.download(k) for k in range(len(b))]
    import lbmhip.batch as batch
    assert _equal(got, several if best["grid"] == batch.GRID_AUTO else single)
    again, same = _batch_run(shape)
    assert again.launch() == shape and _equal(same, got)
    again.set_launch(0, 0)
    assert again.launch() == auto.launch()


@pytest.mark.parametrize("qid,shape,launch", [
    (9, (100, 90), None), (9, (300, 250), None), (9, (1021, 517), None), (9, (2100, 1500), None),
    (17, (512, 512), None), (9, (100, 90), (128, 1, 1, 1)), (9, (128, 64), (128, 1, 1, 1)),
    (13, (40, 30), None)])
def test_timed_runs_count_their_fused_steps(qid, shape, launch):
    """Every step of a run but the collide! that begins it is counted and timed,
    also where one pass holds the whole run; a single-step run that begins with
    collide! and the first fused step in one pass (whole 64 x 8 tiles) leaves
    that step out.  The state is the untimed run's."""
    import lbmhip as L
    q = L.Quadratures[f"D2Q{qid}"]()
    f0 = random_populations(qid, *shape, seed=3)
    one_pass = launch is not None and shape[0] % 64 == 0 and shape[1] % 8 == 0
    for steps in (1, 2, 3, 5, 8, 9, 20):
        a, b = (L.LatticeBoltzmannModel.from_populations(q, f0, L.TRT.fields(0.7, 1.3))
                for _ in (0, 1))
        a.launch = b.launch = launch
        ms, n = L.simulate_timed(a, steps)
        assert n == (max(steps - 2, 0) if one_pass else steps - 1)
        assert ms > 0 or n == 0
        kernel, passes = L.simulate_plan(a, steps)
        assert bool(kernel) == (qid != 13 and steps >= 2 and launch is None)
        assert passes == n if not kernel else (steps + 7) // 8 <= passes <= steps - 1
        L.simulate(b, range(steps))
        assert np.array_equal(a.f_stream.to_numpy(), b.f_stream.to_numpy())
        assert np.array_equal(a.f_collision.to_numpy(), b.f_collision.to_numpy())


def _first_step_model(qid, shape, coll, bcname, force, storage, seed, noise):
    import lbmhip as L
    from lbm_cases import bc_dicts, force_for, to_lbmhip
    q = L.Quadratures[f"D2Q{qid}"]()
    f0 = random_populations(qid, *shape, seed=seed, noise=noise)
    F = force_for(force, *shape)
    cm, taus = {0: (L.SRT(0.8, F), [0.8]), 1: (L.TRT.fields(0.7, 1.3, F), [0.7, 1.3]),
                2: (L.MRT(q, [0.9, 0.75], force=F), [0.9, 0.75])}[coll]
    bcs = bc_dicts(bcname, *shape)

    def model():
        return L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage=storage)

    return model, f0, taus, F, bcs


# whole 64 x 8 tiles whose runs begin with k_fused_first*: with a shape set, and
# without one too long and low for the several-step kernels
FIRST = [((128, 16), (128, 1, 1, 1)), ((64, 8), (64, 4, 1, 1)), ((3392, 8), None)]


@pytest.mark.parametrize("shape,launch", FIRST)
@pytest.mark.parametrize("qid", [4, 5, 9])
@pytest.mark.parametrize("coll", [0, 1, 2])
@pytest.mark.parametrize("bcname,force", [("periodic", "none"), ("couette", "const"),
                                          ("cavity", "field"), ("partial", "none")])
def test_first_step_in_one_pass_bit_exact(oracle_lib, qid, shape, launch, coll, bcname, force):
    """FP64: the run's first step as one pass (collide S_0 into an LDS tile with
    a halo, stream, boundaries, collide) gives the oracle's bits."""
    import lbmhip as L
    model, f0, taus, F, bcs = _first_step_model(qid, shape, coll, bcname, force, "f64",
                                                53 + qid + coll, 2e-3)
    for steps in (2, 5):
        m = model()
        m.launch = launch
        assert L.simulate_timed(m, steps)[1] == steps - 2  # its two steps are one launch
        S, C = f0.copy(order="F"), f0.copy(order="F")
        oracle_lib.simulate(qid, S, C, coll, taus, steps, force=F, bcs=bcs)
        assert np.array_equal(m.f_stream.to_numpy(), S)
        assert np.array_equal(m.f_collision.to_numpy(), C)


@pytest.mark.parametrize("shape,launch", FIRST)
@pytest.mark.parametrize("qid", [4, 5, 9])
@pytest.mark.parametrize("coll", [0, 1])
@pytest.mark.parametrize("bcname,force", [("periodic", "none"), ("couette", "const"),
                                          ("cavity", "field"), ("partial", "none")])
def test_first_step_in_one_pass_f32(qid, shape, launch, coll, bcname, force):
    """FP32 against the two-pass start (collide!, then the fused step): the two
    order a step's operations differently, so each of the two collisions may
    differ by 16 half-ulps of the largest shifted population (the bound of
    test_f32_tracks_oracle), for six steps; a wrong pull, halo or boundary value
    differs by 1e-2 w."""
    import lbmhip as L
    model, f0, *_ = _first_step_model(qid, shape, coll, bcname, force, "f32", 61 + qid, 1e-4)
    one, two = model(), model()
    one.launch = two.launch = launch or (256, 1, 1, 1)
    assert L.simulate_timed(one, 6)[1] == 4
    L.simulate_launch_times(two, 6)
    w = np.asarray(one.quadrature.weights)
    for a, b in ((one.f_stream, two.f_stream), (one.f_collision, two.f_collision)):
        a, b = a.to_numpy(), b.to_numpy()
        G = max(np.abs(b - w).max(), np.abs(f0 - w).max())
        assert np.abs(a - b).max() <= 16 * 7 * 2.0 ** -24 * G


@pytest.mark.parametrize("steps,several", [(2, False), (3, True)])
def test_short_runs_of_batches_of_small_lattices(steps, several):
    """FP32, 512 lattices of 32 x 32 (four nodes computed for one written): two
    steps run one per launch, three in a pass"""
    import lbmhip as L
    f = [random_populations(9, 32, 32, seed=k, noise=1e-2) for k in range(2)]
    out = []
    for launch in (None, (128, 0)):
        b = L.LatticeBatch(L.D2Q9(), [(32, 32)] * 512, [0.7] * 512, [1.3] * 512, storage="f32")
        for k in range(512):
            b.upload(k, f[k % 2])
        if launch:
            b.set_launch(*launch)
        b.simulate(steps)
        out.append([b.download(k) for k in (0, 1, 510, 511)])
    assert _equal(*out) == (not several)
