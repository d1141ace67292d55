"""Strips of deep water over shallows: a sea surface that falls to hpos and below where the
still water is deeper than 3 hpos, and troughs near shallows that it does not dry.  Strips and
tiles evaluate the same face functions in the same order, so a run equals the one of general
tiles alone bit for bit, whatever part of a strip is redone as tiles."""
import numpy as np
import pytest

from conftest import make_problem

pytestmark = pytest.mark.gpu


def _sea(nx, ny, hpos=1.0, ridge=5.0, every=24):
    """4 km of water, ridges `ridge` m deep every `every` rows, depths and hpos in m."""
    pr = make_problem(nx=nx, ny=ny, seed=3, coast=(), fault=False, noise=0.0, seamounts=0, t_sim=1e6)
    D = np.full((ny, nx), 4.0)
    D[12::every, :] = ridge / 1e3
    pr.hmin, pr.H, pr.h, pr.hpos, pr.eps_h = 0.0, D, D.copy(), hpos / 1e3, 1e-8
    return pr


def _run(pr, steps, **kw):
    from thysea import native
    s = native.Solver(pr, **kw)
    t = s.run(max_steps=steps, steps_per_sync=6)["t_final"]
    out = s.state() + (s.field("max_height"), s.field("arrival_times"))
    s.close()
    return t, out


# rows of the troughs after a ridge: on it (below hpos at run time), beside it, further off;
# every strip has one, one strip in some, one in a few
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("off,step,low", [(0, 16, -4.5), (2, 16, -4.5), (10, 16, -4.5), (0, 97, -4.5), (0, 200, -4.9),
                                          (1, 29, -300.0)])
@pytest.mark.parametrize("rows", [0, 5, 16, 19, 40])
def test_troughs(off, step, low, rows, precision):
    pr = _sea(300, 130)
    pr.h[12 + off::24, 7::step] += low / 1e3
    ta, a = _run(pr, 12, precision=precision, strip_rows=rows)
    tb, b = _run(pr, 12, precision=precision, kernel="sweep_general")
    assert ta == tb and np.max(np.abs(a[2])) > 0
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("seed", range(6))
def test_scattered_holes(seed, precision):
    """Low spots anywhere: at the edges of strips, in several places of one, in neighbours."""
    rng = np.random.default_rng(seed)
    pr = _sea(420, 170, ridge=4000.0)
    for _ in range(3 * 2 ** seed):
        y, x = int(rng.integers(0, 170)), int(rng.integers(0, 420))
        D = float(rng.uniform(4e-3, 8e-3))
        pr.H[y, x] = D
        pr.h[y, x] = float(rng.choice([0.3e-3, 0.9e-3, 1.1e-3, D]))
    ta, a = _run(pr, 9, precision=precision, strip_rows=int(rng.integers(9, 64)))
    tb, b = _run(pr, 9, precision=precision, kernel="sweep_general")
    assert ta == tb and all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("precision", [0, 1])
def test_troughs_away_from_shallows_cost_nothing(precision):
    """No cell is shallow at run time: the strips hold, and a step takes as long as on a level
    sea (1.0 expected; a step that redoes every strip takes 4 to 6 times as long)."""
    from thysea import native
    us = []
    for low in (0.0, -4.5):
        pr = _sea(2000, 2000)
        pr.h[22::24, ::16] += low / 1e3
        s = native.Solver(pr, precision=precision)
        t = []
        for _ in range(5):
            s.upload(pr.h, pr.H, pr.qx, pr.qy)
            t.append(s.run(max_steps=6, steps_per_sync=6)["seconds"])
        s.close()
        us.append(float(np.median(t)))
    assert us[1] < 2.0 * us[0], us
