"""Calls at the edge of what the library takes: values that are not finite, contexts without
a state, parameters far from the usual ones.  Against the FP64 oracle, another step kernel or
the call's documented result."""
import numpy as np
import pytest

from conftest import make_problem

pytestmark = pytest.mark.gpu


def _inland(nx=200, ny=60):
    """Land in the eastern half, wide enough for whole tiles of it; returns the problem and
    the depths."""
    pr = make_problem(nx=nx, ny=ny, seed=5, coast=("east",), noise=0.0, fault=False)
    D = pr.H + pr.hmin
    D[:, 90:] = -0.05
    pr.hmin = -0.05
    pr.H = D - pr.hmin
    pr.h = np.maximum(D, 0.0)
    return pr, D


@pytest.mark.parametrize("kernel", ["sweep", "sweep_general", "tile"])
def test_land_that_is_not_finite(kernel):
    """A height beyond FP32's range in the middle of the land: its depth and eta are infinite
    and their sum is no number; the step says so."""
    from thysea import native
    pr, D = _inland()
    pr.H[30, 150] = -1e39
    s = native.Solver(pr, kernel=kernel)
    with pytest.raises(native.ThyError) as e:
        s.step(1e-4)
    assert e.value.code == native.STATUS_CODES["NONFINITE"]
    s.close()


@pytest.mark.parametrize("kernel", ["sweep", "sweep_general", "tile"])
@pytest.mark.parametrize("precision", [0, 1])
def test_without_a_state(kernel, precision):
    """A context without an upload holds dry cells of depth 0: it steps and runs, and stays
    as it is (a run has no wave to wait for, so its first step may reach the end); an upload
    afterwards gives the run of a fresh context."""
    from thysea import native
    pr = make_problem(nx=190, ny=61, seed=9)
    s = native.Solver(pr, upload=False, kernel=kernel, precision=precision)
    assert s.step(1e-4) > 0
    assert s.run(max_steps=7, faults=[])["steps"] >= 1
    assert all(np.all(x == 0) for x in (s.state()[0], s.state()[2], s.state()[3]))
    s.upload(pr.h, pr.H, pr.qx, pr.qy)
    f = native.Solver(pr, kernel=kernel, precision=precision)
    for x in (s, f):
        x.run(max_steps=7)
    assert all(np.array_equal(a, b) for a, b in zip(s.state(), f.state()))
    s.close()
    f.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kernel", ["sweep", "tile"])
def test_infinite_threshold(kernel, precision):
    """hpos infinite: every face takes the WAF flux with blend weight 0, as the limit of the
    formulas says (exp of an infinite argument)."""
    from test_gpu_tiles import _replay
    pr = make_problem(nx=130, ny=44, seed=3)
    pr.hpos = float("inf")
    _replay(pr, 8, precision=precision, kernel=kernel)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("borders", [(1, 1, 1, 1), (1, -1, 2, 2)])
@pytest.mark.parametrize("rows", [1, 4, 5, 6, 7, 8])
def test_every_face_listed_in_rounds(rows, borders, precision):
    """hpos above every depth lists all faces of a tile: a tile of m rows has 57 m + 56 (m + 1)
    of them in the momentum pass, and 508 are taken at a time, those of 4 rows."""
    from test_gpu_tiles import _replay
    assert 4 * 57 + 5 * 56 == 508 and (rows * 57 + (rows + 1) * 56 > 508) == (rows > 4)
    pr = make_problem(nx=185, ny=45, seed=3, borders=borders)
    pr.hpos = 10.0
    _replay(pr, 8, precision=precision, general_rows=rows)


def test_every_face_listed_in_a_batch():
    """A batch's tiles have 8 rows: the same results as alone, with tiles of other heights."""
    from thysea import serving
    pr = make_problem(nx=190, ny=61, seed=9, t_sim=60.0)
    pr.hpos = 10.0
    kw = dict(steps_per_sync=6, keep=[0])
    (ra, a, _), (rb, b) = serving.run_batched([pr], **kw), serving.run_sequential([pr], **kw)
    assert ra[0]["steps"] == rb[0]["steps"] > 6
    assert all(np.array_equal(a[0][k], b[0][k]) for k in ("max_height", "arrival_times"))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kernel", ["sweep", "sweep_general"])
def test_dry_land_and_a_threshold_below_zero(kernel, precision):
    """With hpos below 0 dry cells count as deep; land alone stays as it is all the same."""
    from thysea import native
    pr, D = _inland()
    pr.H[:, :] = 0.0
    pr.h = np.zeros_like(pr.h)
    pr.hpos = -1.0
    s = native.Solver(pr, kernel=kernel, precision=precision)
    a = s.state()
    assert s.step(1e-4) > 0
    s.run(max_steps=3)
    assert all(np.array_equal(x, y) for x, y in zip(a, s.state()))
    s.close()


@pytest.mark.parametrize("t_end", [-1.0, float("nan")])
def test_a_run_that_ends_before_it_starts(t_end):
    """No step and no gauge sample, whatever the series interval."""
    from thysea import native
    pr = make_problem(nx=90, ny=40)
    pr.gauge_pos, pr.series_interval, pr.t_end = np.array([5, 700], np.int32), 0.01, t_end
    s = native.Solver(pr)
    out = s.run(max_steps=5)
    assert out["steps"] == 0 and out["n_samples"] == 0 and out["g_eta"].shape == (0, 2)
    s.close()


@pytest.mark.parametrize("eps_h", [1e100, float("inf")])
@pytest.mark.parametrize("kernel", ["sweep", "tile"])
@pytest.mark.parametrize("precision", [0, 1])
def test_every_cell_dry(precision, kernel, eps_h):
    """eps_h above every depth: the run goes on, and every cell is written as dry."""
    from thysea import native
    pr = make_problem(nx=130, ny=44, seed=3)
    pr.eps_h = eps_h
    s = native.Solver(pr, precision=precision, kernel=kernel)
    assert s.run(max_steps=6)["steps"] >= 1
    assert np.all(np.isfinite(s.state()[0])) and np.all(s.field("eta") == np.float32(-9999))
    s.close()
