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
