"""Runs on the stencils that reach two or three nodes, several steps per pass
(lbm_stage.h), against the oracle.

The pipeline runs from 0.12 to 0.4 million nodes up and writes 112 or 120
columns per block and at least 8 rows per chunk.  The shapes sit at those
edges: whole strips and one column more, ragged sizes, long and low lattices
(17 rows: below three steps' run-in), tall and narrow ones; (300, 200) and
(3001, 15) stay with single steps."""
import numpy as np
import pytest

from lbm_cases import bc_dicts, force_for, to_lbmhip
from test_gpu_multi import _L, _model, _oracle, _populations

pytestmark = pytest.mark.gpu

SHAPES = [(672, 800), (841, 640), (1021, 517), (30001, 17), (224, 4001), (300, 200), (3001, 15)]


def _bcs(name, nx, ny):
    if name == "south":
        return [dict(kind=0, direction=2, xs=(1, nx), ys=(1, ny))]
    if name == "north":
        return [dict(kind=1, direction=0, xs=(1, nx), ys=(1, ny), u=(0.04, 0.0), rho=1.0)]
    if name != "bands":
        return bc_dicts(name, nx, ny)
    # ranges narrower than the walls, a later condition over an earlier one
    return [dict(kind=0, direction=2, xs=(3, nx - 2), ys=(1, 2)),
            dict(kind=1, direction=0, xs=(1, nx), ys=(1, ny), u=(0.04, 0.0), rho=1.0),
            dict(kind=0, direction=0, xs=(5, nx // 2), ys=(ny - 1, ny)),
            dict(kind=0, direction=2, xs=(nx // 2, nx), ys=(2, ny))]


@pytest.mark.parametrize("qid", [13, 17, 21, 37])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("coll,bcname,force,steps", [
    (0, "periodic", "none", 7), (1, "bands", "field", 8), (0, "couette", "const", 5),
    (1, "poiseuille", "const", 2), (1, "cavity", "none", 3), (1, "south", "none", 6),
    (0, "north", "const", 7)])
def test_f64_bit_exact(oracle_lib, qid, shape, coll, bcname, force, steps):
    nx, ny = shape
    f0 = _populations(qid, nx, ny, seed=qid + coll)
    F = force_for(force, nx, ny)
    q, cm, taus = _model(qid, coll, F)
    bcs = _bcs(bcname, nx, ny)
    model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs))
    print(f"stages D2Q{qid} coll {coll} {nx}x{ny} {bcname} {force} {steps} steps", flush=True)
    _L().simulate(model, range(steps))
    S, C = _oracle(oracle_lib, qid, f0, coll, taus, steps, F, bcs)
    assert np.array_equal(model.f_stream.to_numpy(), S)
    assert np.array_equal(model.f_collision.to_numpy(), C)


@pytest.mark.parametrize("qid", [13, 17, 21, 37])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("coll,bcname,force,steps", [
    (0, "periodic", "none", 7), (1, "bands", "field", 8), (1, "poiseuille", "const", 11), (0, "south", "none", 7),
    (1, "north", "none", 7)])
def test_f32_error_no_larger_than_single_steps(oracle_lib, qid, shape, coll, bcname, force, steps):
    """Every step rounds as the single-step kernels do (which the per-launch
    timing entry point keeps): the populations' error against the oracle's
    FP64 run is at most theirs, with a tenth for the scatter of roundings."""
    L = _L()
    nx, ny = shape
    f0 = _populations(qid, nx, ny, seed=11, noise=1e-4)
    F = force_for(force, nx, ny)
    q, cm, taus = _model(qid, coll, F)
    bcs = _bcs(bcname, nx, ny)
    print(f"stages f32 D2Q{qid} coll {coll} {nx}x{ny} {bcname} {force}", flush=True)
    many = L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage="f32")
    L.simulate(many, range(steps))
    one = L.LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs), storage="f32")
    L.simulate_launch_times(one, steps)
    S, C = _oracle(oracle_lib, qid, f0, coll, taus, steps, F, bcs)
    for a, b, ref in ((many.f_stream, one.f_stream, S), (many.f_collision, one.f_collision, C)):
        ea, eb = (np.linalg.norm(x.to_numpy() - ref) for x in (a, b))
        assert ea <= 1.1 * eb, (ea, eb)


@pytest.mark.parametrize("qid", [13, 17, 21, 37])
@pytest.mark.parametrize("shape", [(672, 800), (1021, 517), (30001, 17)])
@pytest.mark.parametrize("coll,bcname,steps", [(0, "couette", 6), (1, "poiseuille", 8),
                                               (1, "couette", 9)])
def test_f64_later_passes_between_two_walls_bit_exact(oracle_lib, qid, shape, coll, bcname, steps):
    """passes of three steps (D2Q13 and D2Q17) that pull their first one"""
    nx, ny = shape
    f0 = _populations(qid, nx, ny, seed=qid + 5 * coll)
    q, cm, taus = _model(qid, coll, None)
    bcs = _bcs(bcname, nx, ny)
    model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs))
    print(f"stages later D2Q{qid} {nx}x{ny} {bcname} {steps} steps", flush=True)
    _L().simulate(model, range(steps))
    S, C = _oracle(oracle_lib, qid, f0, coll, taus, steps, None, bcs)
    assert np.array_equal(model.f_stream.to_numpy(), S)
    assert np.array_equal(model.f_collision.to_numpy(), C)


@pytest.mark.parametrize("qid", [13, 17, 21, 37])
@pytest.mark.parametrize("shape", [(672, 800), (1021, 517), (30001, 17)])
@pytest.mark.parametrize("direction", [0, 2])
@pytest.mark.parametrize("steps", [3, 8])
def test_f64_one_ranged_wall_bit_exact(oracle_lib, qid, shape, direction, steps):
    """one wall over a part of its row, a later condition of the same wall over
    another part; passes of up to three steps"""
    nx, ny = shape
    f0 = _populations(qid, nx, ny, seed=qid + direction)
    q, cm, taus = _model(qid, 1, None)
    ys = (1, 2) if direction == 2 else (ny - 2, ny)
    bcs = [dict(kind=0, direction=direction, xs=(5, nx // 2), ys=ys),
           dict(kind=0, direction=direction, xs=(nx // 3, nx - 60), ys=(1, ny))]
    model = _L().LatticeBoltzmannModel.from_populations(q, f0, cm, to_lbmhip(bcs))
    print(f"stages one wall {direction} D2Q{qid} {nx}x{ny} {steps} steps", flush=True)
    _L().simulate(model, range(steps))
    S, C = _oracle(oracle_lib, qid, f0, 1, taus, steps, None, bcs)
    assert np.array_equal(model.f_stream.to_numpy(), S)
    assert np.array_equal(model.f_collision.to_numpy(), C)
