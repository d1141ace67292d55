"""Okada sources off the beaten form: vertical faults, pure strike or dip slip, a fault whose
edge lines pass through cells, and the pass that adds the displacement at once against the
one that keeps the field; against the FP64 oracle.

Tolerance 1e-10 of the peak, as for the thrust source: the sums cancel terms some 1e4 times
the far field, each rounded to 1e-16."""
import numpy as np
import pytest

from conftest import make_problem, rel_linf

pytestmark = pytest.mark.gpu

FORMS = [dict(dip=90.0, rake=0.0), dict(dip=90.0, rake=90.0), dict(dip=89.0, rake=40.0), dict(dip=20.0, rake=0.0),
         dict(dip=20.0, rake=180.0), dict(dip=35.0, rake=90.0, strike=0.0), dict(dip=35.0, rake=270.0, strike=90.0)]


@pytest.mark.parametrize("form", FORMS)
def test_okada_forms(form):
    import oracle as O
    from thysea import native
    pr = make_problem(nx=96, ny=80)
    # centroid on a cell: for strike 0 and 90 the plane's axes run through cells
    f = dict(dict(time=0.0, lon_c=float(pr.lon[40]), lat_c=float(pr.lat[37]), depth_c=28.0, length=80.0, width=40.0,
                  strike=33.0, dip=30.0, rake=90.0, slip=3.0), **form)
    s, o = native.Solver(pr), O.OracleSim(pr)
    dg, do = s.okada(f, want_def=True), o.okada(f, want_def=True)
    scale = float(np.max(np.abs(do)))
    assert scale > 0 and np.array_equal(np.isnan(dg), np.isnan(do))
    assert rel_linf(dg, do, scale) < 1e-10
    # the same source again without the field, uncropped and cropped: FP32 state, so
    # rounding of eta and depth (a 4 km depth: 2.4e-7 km) bounds the difference
    for crop, value in ((0, 0.0), (2, 0.2 * scale)):
        a, b = native.Solver(pr), native.Solver(pr)
        a.okada(f, crop, value)
        b.okada(f, crop, value, want_def=True)
        assert all(np.array_equal(p, q) for p, q in zip(a.state(), b.state()))
        a.close()
        b.close()
    s.close()
