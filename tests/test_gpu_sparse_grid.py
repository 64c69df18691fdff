"""A grid that is mostly empty: whole blocks of tiles without particles beside
ones with a few, the state equal to the oracle's (FP32-mixed within 1e-4)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("side,capacity", [(2.0, None), (2.0, 120000), (4.6, None)])  # 0.5, 5.6 million cells
def test_scattered_clusters(side, capacity, prec):
    from oracle.pyoracle import Oracle
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(side, side, side), column=(0.1, 0.1, 0.1), dx=0.01, name="sparse"), particles=False,
               incidence=False)
    rng = np.random.default_rng(6)
    at = np.concatenate([[[0.05, 0.05, 0.05], [side - 0.05] * 3], rng.uniform(0.05, side - 0.05, (30, 3))])
    coord = np.concatenate([c + rng.uniform(-0.03, 0.03, (60, 3)) for c in at])
    n = len(coord)
    dens = 1000.0 * (1.0 + rng.uniform(-1e-3, 1e-3, n))
    kw = dict(vel=rng.normal(0.0, 0.5, (n, 3)), dens=dens, pres=tb.case.bulk / 1000.0 * (dens - 1000.0),
              mass=np.full(n, 1e-3))
    o = Oracle(tb, coord=coord, semi=False, **kw)
    d = rt.SphContext(tb, precision=prec, capacity=capacity or n, semi=False)
    d.upload(coord=coord, **kw)
    for x in (o, d):
        x.preloop()
        x.step(5)
    s, r = d.state(), o.state()
    d.close()
    for f in ("coord", "vel", "acc", "dens", "pres", "dden", "vpres"):
        tol = 1e-4 * np.abs(r[f]).max() if prec else 0.0
        assert np.abs(s[f] - r[f]).max() <= tol, f
