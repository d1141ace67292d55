"""General tiles of the row sweep at their edges: tiles of 1 to 8 rows, segments of one
column and of whole width, every face on the work list (more than one round of results),
land, and strips redone as tiles; against the FP64 oracle with its dt replayed.

Tolerance: the one of the other oracle comparisons, 1e-4 of the peak in FP32 and 1e-9 in
FP64 (each step rounds a cell a few dozen times, 6e-8 or 1e-16 relative each; tens of
steps stay orders below)."""
import numpy as np
import pytest

from conftest import make_problem, rel_linf

pytestmark = pytest.mark.gpu


def _replay(pr, steps, **kw):
    import oracle as O
    from thysea import native
    g, o = native.Solver(pr, **kw), O.OracleSim(pr)
    for f in pr.faults:
        g.okada(f)
        o.okada(f)
    dt = o.initial_dt()
    for _ in range(steps):
        dn = o.step(dt)
        g.step(dt)
        dt = dn
    a, b = g.state(), o.state()
    g.close()
    peak = max(float(np.max(np.abs(b[0] - b[1] - pr.hmin))), 1e-30)
    tol = 1e-9 if kw.get("precision") else 1e-4
    wet = b[0] > pr.eps_h
    assert np.array_equal(a[0] > pr.eps_h, wet)
    assert rel_linf((a[0] - a[1])[wet], (b[0] - b[1])[wet], peak) < tol
    assert rel_linf(a[2], b[2], peak) < tol and rel_linf(a[3], b[3], peak) < tol


# ny modulo the tile rows 1, 2, 3, 4, 7, 0; nx one column past a segment, exactly one, ragged
@pytest.mark.parametrize("nx,ny", [(57, 9), (56, 18), (113, 27), (61, 36), (170, 47), (112, 64)])
@pytest.mark.parametrize("general_rows", [1, 3, 4, 8])
def test_tile_heights(nx, ny, general_rows):
    _replay(make_problem(nx=nx, ny=ny, seed=nx + ny), 12, general_rows=general_rows, strip_rows=8)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("borders", [(1, 1, 1, 1), (-1, -1, -1, -1), (1, -1, 2, 2)])
def test_every_face_listed(borders, precision):
    """hpos above every depth: no face takes the deep form, so a tile lists all of them."""
    pr = make_problem(nx=130, ny=44, seed=3, borders=borders)
    pr.hpos = 10.0
    _replay(pr, 8, precision=precision)


@pytest.mark.parametrize("lake", [False, True])
def test_land(lake):
    """Whole tiles of dry land beside water, and a lake one cell wide in the land."""
    pr = make_problem(nx=200, ny=60, seed=5, coast=("east",), noise=0.0)
    land = np.zeros((60, 200), bool)
    land[:, 90:] = True
    if lake:
        land[30, 150] = False
    D = np.where(land, -0.05, pr.H + pr.hmin)
    pr.hmin = -0.05
    pr.H = D - pr.hmin
    pr.h = np.maximum(D, 0.0)
    _replay(pr, 12)
    # and the dry cells' arrival (their eta_ini is a marker) as the other step kernel has it
    from thysea import native
    out = []
    for kernel in ("sweep", "tile"):
        s = native.Solver(pr, kernel=kernel)
        s.run(max_steps=6)
        out.append((s.field("arrival_times"), s.field("max_height")))
        s.close()
    assert np.array_equal(out[0][0] < 0, out[1][0] < 0) and np.array_equal(out[0][1] < -9000, out[1][1] < -9000)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", [(700, 300), (300, 130), (90, 45)])
def test_tiles_of_mixed_heights(nx, ny, precision):
    """Tiles made lower along the coast (the default) against tiles of one height, of eight
    rows and of five: the same faces and the same sums, bit for bit."""
    from thysea import native
    pr = make_problem(nx=nx, ny=ny, seed=nx, coast=("north", "east"))
    out = []
    for rows in (0, 8, 5):
        s = native.Solver(pr, general_rows=rows, precision=precision)
        s.run(max_steps=18, steps_per_sync=6)
        out.append(s.state() + (s.field("max_height"), s.field("arrival_times")))
        s.close()
    for o in out[1:]:
        for x, y in zip(out[0], o):
            assert np.array_equal(x, y)
