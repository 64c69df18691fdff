"""Integer positions in 2D: the plane's cells set their unit, whatever the side
of the single cell row in y, and particles whole wraps of the positions apart in
y are no neighbours.  Lists equal the oracle's; fields at the bars of the other
2D tests (FP64 1e-11, FP32-mixed 1e-4 of each field's largest value)."""
import numpy as np
import pytest

from sphera_amd import case2d
from tests.test_gpu_2d import FIELDS, FP32_TOL, FP64_REL_TOL, SMALL, _jitter2d, _lists_equal, _rel

pytestmark = pytest.mark.gpu


def _held(tb, prec, coord, row):
    """row: the y cell side on the device (the oracle's row holds every particle)."""
    from oracle.pyoracle import Oracle
    from sphera_amd import runtime as rt
    tb.grid.extr_lo[1] = -1.0e4
    tb.grid.dcd[1] = 2.0e4
    o = Oracle(tb, coord=coord)
    o.preloop()
    tb.grid.dcd[1] = row
    d = rt.SphContext(tb, precision=prec)
    d.upload(coord=coord)
    d.preloop()
    _lists_equal(d, o)
    d.step(8)
    o.step(8)
    _lists_equal(d, o)
    s, r = d.state(), o.state()
    d.close()
    for f in FIELDS:
        assert _rel(s[f], r[f]) <= (FP32_TOL[f] if prec else FP64_REL_TOL), f
    return r


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("row", [1.0, 1000.0, 1.0e6])
def test_wide_row(row, prec):
    tb = case2d.build(case2d.DamBreak2D(**SMALL))
    _held(tb, prec, _jitter2d(tb.particles["coord"], tb.case.dx), row)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("wraps", [0, 1, -3])
def test_particles_apart_in_y(wraps, prec):
    """A third of the particles whole wraps (16 cells) away in y, all of them
    jittered in y."""
    tb = case2d.build(case2d.DamBreak2D(**SMALL))
    side = max(tb.grid.dcd[0], tb.grid.dcd[2])
    coord = _jitter2d(tb.particles["coord"], tb.case.dx)
    rng = np.random.default_rng(4)
    coord[:, 1] += rng.uniform(-0.2, 0.2, len(coord)) * tb.case.dx
    coord[::3, 1] += 16.0 * side * wraps
    _held(tb, prec, coord, tb.grid.dcd[0])
