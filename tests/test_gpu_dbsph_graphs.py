"""Captured DB-SPH steps and wall kinematics set after the capture: the records
and their buffer change between two solves of one context, so the steps are
captured again.  The replayed steps equal a new context's eager steps."""
import numpy as np
import pytest

from sphera_amd.case import build
from tests.test_gpu_dbsph import DBF, FIELDS, _case

pytestmark = pytest.mark.gpu

STILL = [(0.0,) * 7, (100.0,) + (0.0,) * 6]
MOVING = [(0.0,) * 7, (0.01, 0.5, 0.0, 0.0, 0.0, 0.0, 1.0), (100.0, 0.5, 0.0, 0.0, 0.0, 0.0, 1.0)]


def _set(d, rec):
    from sphera_amd import runtime as rt
    k = np.array(rec, np.float64).reshape(-1, 7)
    c = np.array([0.1, 0.05, 0.0])
    d._check(d.L.sph_dbsph_kinematics(d.h, len(k), rt._pd(k), rt._pd(c)), "sph_dbsph_kinematics")


@pytest.mark.parametrize("first,then", [([], MOVING), (STILL, MOVING), (STILL, [])])
def test_kinematics_after_capture(first, then):
    from sphera_amd import runtime as rt
    tb = build(_case())
    d = rt.SphContext(tb, precision=rt.FP64)
    e = rt.SphContext(tb, precision=rt.FP64)
    _set(d, first)
    d.upload()
    d.preloop()
    print(f"[gpu] {len(first)} records, then {len(then)}", flush=True)
    for _ in range(3):  # the walls rest: a new solve finds them where they were
        d.step_graph(1)
    d.sync()
    d.upload()
    for c in (d, e):
        _set(c, then)
    e.upload()
    for c in (d, e):
        c.preloop()
    for _ in range(4):
        d.step_graph(1)
    d.sync()
    e.step(4)
    s, t, b, r = d.state(), e.state(), d.dbsph_state(), e.dbsph_state()
    d.close()
    e.close()
    assert s["time"] == t["time"]
    for f in FIELDS:
        assert np.array_equal(s[f], t[f]), f
    for f in DBF:
        if f != "wall_wet":  # wet once, wet for good
            assert np.array_equal(b[f], r[f]), f
