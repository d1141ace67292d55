"""Fields large enough to be read in chunks by several threads: every cell arrives in its
place, with the library's caches filled and emptied, and read from two threads at once.

Tolerance: a field is one FP32 rounding (6e-8) away from a depth times the problem's scale,
which the state gives in FP64; 1e-6 of the peak."""
import threading

import numpy as np
import pytest

from conftest import make_problem

pytestmark = pytest.mark.gpu


def _check(s, pr, scale, out):
    h, H, _, _ = s.state()
    D = H + pr.hmin
    for name, want in (("deformed_bathy", D * scale), ("eta", np.where(h < pr.eps_h, -9999.0, (h - D) * scale))):
        got = s.field(name)
        wet = want > -9000
        out.append(np.array_equal(got > -9000, wet) and
                   np.max(np.abs(got - want)[wet]) <= 1e-6 * np.max(np.abs(D * scale)))


# below the chunked size; whole chunks (2048 x 1024 cells of 4 bytes each) and ragged ones
@pytest.mark.parametrize("nx,ny", [(1400, 1200), (2048, 1024), (2047, 1031), (2903, 2111)])
@pytest.mark.parametrize("trimmed", [False, True])
def test_every_cell_in_its_place(nx, ny, trimmed):
    from thysea import native
    pr = make_problem(nx=nx, ny=ny, seed=3, coast=("north",), lat0=-30.0)
    solvers = [native.Solver(pr, precision=p) for p in (0, 1)]
    if trimmed:
        native.lib().thy_release_cached()
    scale = solvers[0].params.H
    out = []
    threads = [threading.Thread(target=_check, args=(s, pr, scale, out)) for s in solvers]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in solvers:
        s.close()
    assert out == [True] * 4
