"""lbm_simulate_plan: which kernel a run takes and in how many passes (the
rules need no GPU)."""
import ctypes

import pytest

import lbmhip._lib as lib

SRT, TRT, MRT = 0, 1, 2


def plan(qid, storage, coll, nx, ny, nsteps, walls=(), launch=(0, 0, 0, -1)):
    """walls: directions (0 N, 1 E, 2 S, 3 W) of bounce-back walls"""
    arr = (lib.LbmBC * max(1, len(walls)))()
    for k, d in enumerate(walls):
        arr[k].kind, arr[k].direction = 0, d
        arr[k].x0, arr[k].x1, arr[k].y0, arr[k].y1 = 1, nx, 1, ny
    kernel, passes = ctypes.c_char_p(), ctypes.c_int64()
    rc = lib.lib().lbm_simulate_plan(qid, lib.STORAGES[storage], coll, nx, ny, arr, len(walls),
                                     *launch, nsteps, ctypes.byref(kernel), ctypes.byref(passes))
    assert rc == 0, lib.lib().lbm_last_error()
    return kernel.value.decode(), passes.value


@pytest.mark.parametrize("storage,passes", [("f64", 4), ("f32", 4), ("f16neq", 5), ("bf16neq", 5)])
def test_passes_of_twenty_steps(storage, passes):
    assert plan(9, storage, TRT, 4096, 4096, 20) == ("k_march", passes)


def test_single_steps_are_timed_after_the_first_launch():
    assert plan(9, "f16dev", TRT, 4096, 4096, 20) == ("", 18)  # whole 64 x 8 tiles
    assert plan(9, "f16dev", TRT, 4095, 4096, 20) == ("", 19)
    assert plan(37, "f64", MRT, 2048, 1024, 20) == ("", 19)
    assert plan(9, "f64", TRT, 64, 64, 1) == ("", 0)
    assert plan(9, "f64", TRT, 64, 64, 0) == ("", 0)


@pytest.mark.parametrize("args,kernel", [
    ((9, "f64", TRT, 168, 160, 8), "k_tile"), ((9, "f64", TRT, 169, 160, 8), "k_block"),
    ((9, "f64", MRT, 1500, 1500, 8), "k_block"), ((9, "f64", SRT, 2048, 1500, 8), "k_march"),
    ((9, "f32", SRT, 2048, 1500, 8), "k_block"), ((5, "f32", SRT, 4000, 3000, 8), "k_march"),
    ((9, "f64", TRT, 31, 2501, 8), ""), ((17, "f64", TRT, 600, 500, 8), "k_stages"),
    ((17, "f64", TRT, 100, 90, 8), ""), ((17, "f64", MRT, 600, 500, 8), "")])
def test_kernel_of_a_run(args, kernel):
    assert plan(*args)[0] == kernel


@pytest.mark.parametrize("walls,least", [((), 800000), ((0, 2), 1200000), ((2,), 1200000),
                                         ((1,), 1800000), ((0, 1, 2, 3), 1800000)])
def test_16_bit_lines_follow_the_walls(walls, least):
    ny = least // 1000
    assert plan(9, "f16neq", TRT, 1000, ny, 3, walls)[0] == "k_march"
    assert plan(9, "f16neq", TRT, 1000, ny - 1, 3, walls)[0] == ""
    assert plan(9, "f16neq", TRT, 1000, 2 * ny, 2, walls)[0] == "k_march"
    assert plan(9, "f16neq", TRT, 1000, 2 * ny - 1, 2, walls)[0] == ""
    assert plan(9, "f16neq", TRT, 128, 6250, 3, walls)[0] == "k_march"
    assert plan(9, "f16neq", TRT, 128, 20000, 2, walls)[0] == ""


def test_two_steps_on_whole_tiles():
    for nx, ny, kernel in ((4096, 4096, ""), (4095, 4096, "k_march"), (64, 8000, ""),
                           (6400, 64, ""), (1536, 1024, "k_block"), (128, 128, "k_tile")):
        assert plan(9, "f64", TRT, nx, ny, 2)[0] == kernel
        assert plan(9, "f64", TRT, nx, ny, 3)[0] in ("k_tile", "k_block", "k_march")


def test_plan_errors():
    L, bc = lib.lib(), (lib.LbmBC * 1)()
    for *args, steps in ((10, 0, 0, 8, 8, bc, 0, 3), (9, 99, 0, 8, 8, bc, 0, 3),
                         (9, 0, 3, 8, 8, bc, 0, 3), (9, 0, 0, 0, 8, bc, 0, 3),
                         (9, 0, 0, 8, 8, None, 1, 3), (9, 0, 0, 8, 8, bc, 0, -1)):
        assert L.lbm_simulate_plan(*args, 0, 0, 0, -1, steps, None, None) < 0
    assert L.lbm_simulate_plan(9, 0, 0, 8, 8, bc, 0, 96, 0, 0, -1, 3, None, None) < 0


def test_plan_of_a_launch_shape():
    assert plan(9, "f32", TRT, 300, 250, 9, launch=(256, 1, 1, 1)) == ("", 8)
    assert plan(9, "f32", TRT, 320, 240, 9, launch=(256, 1, 1, 0)) == ("", 7)
    assert plan(9, "f32", TRT, 300, 250, 9, launch=(128, 1, 1, -1)) == ("", 8)
    assert plan(9, "f32", TRT, 300, 250, 9, launch=(256, 1, 1, -1))[0] == "k_block"


@pytest.mark.parametrize("qid,storage", [(4, "f64"), (5, "f32"), (9, "f32"), (9, "f16neq"),
                                         (13, "f32")])
def test_rows_beyond_32_bit_offsets_keep_single_steps(qid, storage):
    """the several-step kernels refuse rows of 2^27 nodes; the single-step ones
    take them"""
    assert plan(qid, storage, TRT, 2 ** 27 - 2, 15 if qid < 13 else 16, 9)[0] != ""
    assert plan(qid, storage, TRT, 2 ** 27, 15 if qid < 13 else 16, 9) == ("", 8)
    assert plan(qid, storage, TRT, 2 ** 27, 1, 9) == ("", 8)


@pytest.mark.parametrize("n,storage,steps,kernel,passes,per_pass", [
    (4096, "f64", 20, "k_march", 4, 5.0), (4096, "f32", 20, "k_march", 4, 5.0),
    (4096, "f32", 5000, "k_march", 834, 5000 / 834), (1024, "f64", 20, "k_block", None, None),
    (4096, "f16dev", 20, "", 18, 1.0), (4095, "f16dev", 20, "", 19, 1.0)])
def test_bench_prices_the_passes_that_run(n, storage, steps, kernel, passes, per_pass):
    """the benchmark's kernel, time of a pass and steps per pass follow the plan
    of the run at hand"""
    from types import SimpleNamespace

    import bench
    import lbmhip as L
    model = SimpleNamespace(quadrature=L.D2Q9(), boundary_conditions=[], launch=None,
                            collision_model=L.TRT.fields(0.6, 1.3),
                            f_stream=SimpleNamespace(storage=storage, nx=n, ny=n))
    counted = passes if not kernel else steps - 1
    got = bench.pass_figures(L, model, steps, 7.0, counted)
    assert got[0] == kernel
    if passes:
        assert got[1:] == pytest.approx((7.0 / passes, per_pass))
    assert got[1] * (steps if kernel else counted) / got[2] == pytest.approx(7.0)
    assert bench.pass_figures(L, model, 1, 0.005, 0) == ("", 0.0, 0.0)


def test_bench_traffic_belongs_to_the_kernel_and_size():
    import bench
    march = bench.traffic_for("f64", 4096, "k_march")
    assert march > 1.1 * bench.traffic_for("f64", 4096, "") > 0
    assert bench.traffic_for("f64", 1024, "k_block") is None
