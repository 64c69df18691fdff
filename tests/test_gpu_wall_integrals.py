"""FP64 wall integrals by four lanes a pair against the oracle: a column in a
corner (rings inside, across and outside the faces), and a quadrature table
whose rings do not share their weight (the direction-by-direction form)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("tank", [(0.3, 0.1, 0.2), (0.062, 0.055, 0.07)])
def test_integrals_match_oracle(tank, even):
    from oracle.pyoracle import Oracle
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=tank, column=(0.06, 0.05, 0.06), dx=0.01, name="corner"))
    if not even:
        tb.bitab = tb.bitab.copy()
        tb.bitab[37, 3] *= 1.0 + 1.0e-7
    rng = np.random.default_rng(5)
    c = tb.particles["coord"]
    coord = c + rng.uniform(-0.3, 0.3, c.shape) * tb.case.dx
    o = Oracle(tb, coord=coord)
    o.preloop()
    o.step(8)
    d = rt.SphContext(tb, precision=rt.FP64)
    d.upload(coord=coord)
    d.preloop()
    d.step(8)
    so, sd = o.state(), d.state()
    d.close()
    for f in ("coord", "vel", "acc", "dens", "pres", "dden", "vpres"):
        assert np.array_equal(so[f], sd[f]), f
