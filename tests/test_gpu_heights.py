"""Heights of strips and tiles that a caller asks for are the ones that run.  No result depends
on them, so they show in the time of a step: heights are chosen that cost several times the
default's (a strip is a chain of rows, 0.5 us each and more), and the bounds are half of that."""
import numpy as np
import pytest

from conftest import make_problem

pytestmark = pytest.mark.gpu


def _us(s, n=48, reps=5):
    """Us a step of a run in progress, the median of reps."""
    return float(np.median([s.run_more(n)["seconds"] for _ in range(reps)])) / n * 1e6


def _solver(pr, **kw):
    from thysea import native
    s = native.Solver(pr, **kw)
    s.run(max_steps=48, steps_per_sync=48)
    return s


def test_tall_strips_on_a_small_grid():
    """One strip of deep water from border to border, where the default has strips of 8 rows."""
    pr = make_problem(nx=1000, ny=800, seed=9, coast=(), seamounts=0, t_sim=1e6)
    a, b = _solver(pr), _solver(pr, strip_rows=788)
    assert _us(b) > 4 * _us(a)
    assert all(np.array_equal(x, y) for x, y in zip(a.state(), b.state()))


def test_autotune_starts_from_the_heights_in_use():
    """FP64 500x400 without a coast is fastest with strips lower than any the tuner tries (3 rows
    against 8: a chain of 11 rows against 16, 14 us against 17); they stay."""
    pr = make_problem(nx=500, ny=400, seed=9, coast=(), seamounts=0, t_sim=1e6)
    s = _solver(pr, precision=1, strip_rows=3)
    before = s.state()
    assert s.autotune(5)[0] == 3
    assert all(np.array_equal(x, y) for x, y in zip(before, s.state()))


def test_tuned_heights_survive_an_upload():
    """A height that autotune replaced does not come back with the next state."""
    pr = make_problem(nx=1000, ny=800, seed=9, coast=(), seamounts=0, t_sim=1e6)
    s = _solver(pr, strip_rows=788)
    slow = _us(s)
    rows, _ = s.autotune(5)
    assert rows < 100 and _us(s) < slow / 4
    s.upload(pr.h, pr.H, pr.qx, pr.qy)
    s.run(max_steps=48, steps_per_sync=48)
    assert _us(s) < slow / 4
    assert s.autotune(5)[0] < 100


def test_tile_height_in_a_batch():
    """Tiles of one row load nine for it, and are eight times as many."""
    from thysea import serving
    pr = make_problem(nx=700, ny=600, seed=9, coast=("north", "east"), t_sim=120.0)
    us, res = {}, {}
    for rows in (0, 8, 1):
        kw = dict(kernel="sweep_general", general_rows=rows)
        gpu = []
        for _ in range(3):
            rec, out, g = serving.run_batched([pr] * 8, steps_per_sync=24, keep=range(8), solver_kw=kw)
            gpu.append(g)
        us[rows], res[rows] = float(np.median(gpu)), out
    assert us[1] > 2 * us[8] and us[0] < 1.5 * us[8], us
    for i in range(8):
        assert np.array_equal(res[1][i]["max_height"], res[8][i]["max_height"])
