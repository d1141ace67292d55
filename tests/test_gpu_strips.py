"""Deep-water strips at their edges: heights of every remainder of the row loop, and strips
whose depth check fails in mid-ocean and which are then redone as tiles.  Strips and tiles
evaluate the same face functions in the same order, so the run equals the one of general
tiles alone bit for bit."""
import numpy as np
import pytest

from conftest import make_problem

pytestmark = pytest.mark.gpu


def _run(pr, steps, **kw):
    from thysea import native
    s = native.Solver(pr, **kw)
    s.run(max_steps=steps, steps_per_sync=6)
    h, H, qx, qy = s.state()
    out = h - H, qx, qy, s.field("max_height"), s.field("arrival_times")
    s.close()
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8, 31, 40])
def test_strip_heights(rows, precision):
    pr = make_problem(nx=190, ny=61, seed=9, coast=())
    a = _run(pr, 18, precision=precision, strip_rows=rows)
    b = _run(pr, 18, precision=precision, kernel="sweep_general")
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("spot", [(40, 90), (24, 59), (25, 60)])
def test_failed_strips(spot, precision):
    """hpos a quarter of the least depth, and a hole in the surface down to half of hpos."""
    pr = make_problem(nx=260, ny=90, seed=9, coast=(), fault=False)
    D = pr.H + pr.hmin
    pr.hpos = float(D.min()) / 4
    y, x = spot
    h = D.copy()
    h[y:y + 2, x:x + 2] = pr.hpos / 2
    pr.h = h
    a = _run(pr, 12, precision=precision, strip_rows=16)
    b = _run(pr, 12, precision=precision, kernel="sweep_general")
    assert np.all(np.isfinite(a[0])) and np.max(np.abs(a[1])) > 0
    for p, q in zip(a, b):
        assert np.array_equal(p, q)


def test_rows_beyond_the_pole():
    """A grid that runs past the pole has rows of negative area and length, whose wave speeds
    sum to less than the guard of a cell's dt: such cells set no dt."""
    pr = make_problem(nx=300, ny=200, seed=9, coast=(), lat0=85.0)
    a = _run(pr, 7)
    b = _run(pr, 7, kernel="sweep_general")
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("nx,ny,precision", [(2803, 2701, 0), (1997, 1901, 1)])
def test_strips_in_reverse_order(nx, ny, precision):
    """State above the size from which every other step walks the strips backwards."""
    pr = make_problem(nx=nx, ny=ny, seed=9, coast=("north",))
    a = _run(pr, 7, precision=precision)
    b = _run(pr, 7, precision=precision, kernel="sweep_general")
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("n", [1, 3, 5])
def test_batch_in_reverse_order(n):
    """Batches below and above the size from which every other step walks the strips
    backwards, the first scenario without a coast, against each scenario alone."""
    from thysea import serving
    prs = [make_problem(nx=1450 + 57 * i, ny=1310 - 31 * i, seed=9 + i, coast=("north", "east") if i else (), t_sim=60.0)
           for i in range(n)]
    rec_b, res_b, _ = serving.run_batched(prs, steps_per_sync=6, keep=range(n))
    rec_s, res_s = serving.run_sequential(prs, steps_per_sync=6, keep=range(n))
    for i in range(n):
        assert rec_b[i]["steps"] == rec_s[i]["steps"] > 6
        for key in ("max_height", "arrival_times"):
            assert np.array_equal(res_b[i][key], res_s[i][key]), (i, key)
