"""DB-SPH launch forms: lanes per particle by capacity (eight, four) and the
list kernel's block size by its LDS (long neighbour lists: one wavefront or one
particle a block) give the same bits, and the oracle's."""
import numpy as np
import pytest

from sphera_amd.case import build
from tests.test_gpu_dbsph import COMBINED, DBF, FIELDS, _case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small():
    from oracle.pyoracle import Oracle
    tb = build(_case(COMBINED))
    rng = np.random.default_rng(3)
    c = tb.particles["coord"]
    coord = c + rng.uniform(-0.01, 0.01, c.shape) * tb.case.dx
    o = Oracle(tb, coord=coord)
    o.preloop()
    o.step(12)
    return tb, coord, o.state(), o.dbsph_state()


@pytest.mark.parametrize("capacity,nmaxpartj", [(None, None), (19999, None), (20000, None), (20000, 10000), (60000, 60000)])
def test_dbsph_forms(small, capacity, nmaxpartj):
    from sphera_amd import runtime as rt
    tb, coord, so, do = small
    keep = tb.scalars["nmaxpartj"]
    tb.scalars["nmaxpartj"] = nmaxpartj or keep
    try:
        d = rt.SphContext(tb, precision=rt.FP64, capacity=capacity)
    finally:
        tb.scalars["nmaxpartj"] = keep
    d.upload(coord=coord)
    d.preloop()
    d.step(12)
    s, b = d.state(), d.dbsph_state()
    d.close()
    for f in FIELDS:
        assert np.array_equal(s[f], so[f]), f
    for f in DBF:
        assert np.array_equal(b[f], do[f]), f
