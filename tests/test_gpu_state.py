"""State download in pg order: a permuted upload comes back row for row, and
where a sort removed more particles than it renumbers (ids with gaps) the rows
are the remaining particles by ascending id."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("outside", [0, 5000])
def test_download_rows(outside, prec):
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.3, 0.2, 0.2), column=(0.3, 0.2, 0.2), dx=0.01, name="cloud"))
    rng = np.random.default_rng(outside + 1)
    n = 1237 + outside
    coord = rng.uniform(0.002, np.array([0.298, 0.198, 0.198]), (n, 3))
    out = rng.permutation(n)[:outside]
    coord[out] += 10.0
    vel = rng.normal(0.0, 1.0, (n, 3))
    dens, pres = rng.uniform(990.0, 1010.0, n), rng.uniform(0.0, 10.0, n)
    d = rt.SphContext(tb, precision=prec, capacity=n + 5, semi=False)
    d.upload(coord=coord, vel=vel, dens=dens, pres=pres, mass=np.full(n, 1e-3))
    st = d.state()
    d.close()
    keep = np.setdiff1d(np.arange(n), out)
    assert np.array_equal(st["ids"], keep)
    for f, a in (("coord", coord), ("vel", vel), ("dens", dens), ("pres", pres)):
        assert np.array_equal(st[f], a[keep]), f
    for f in ("acc", "dden", "vpres"):
        assert not st[f].any(), f
