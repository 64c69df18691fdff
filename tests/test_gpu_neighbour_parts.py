"""Cells with more candidates than a wavefront's registers hold: they are taken
in parts.  Candidate counts around the parts' edges, more than 64 particles in a
cell, lists cut at NMAXPARTJ inside the first part, in a later one and at the
edges of eight, lists of LDS slots (one mass) and of indices (FP64 with two).
Lists equal the oracle's; the next steps, which read what fills a list up, too
(FP64; FP32-mixed within 1e-4 of each field's largest value, velocity and
pressure sums of a cluster being large)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("coord", "vel", "acc", "dens", "pres", "dden", "vpres")


@pytest.mark.parametrize("prec,masses", [(0, 1), (0, 2), (1, 1), (1, 2)])
@pytest.mark.parametrize("m,cut", [(641, 0), (704, 24), (768, 300), (769, 301), (1024, 7), (1025, 8), (1280, 100),
                                   (1281, 9), (2400, 0), (2400, 163), (3300, 1000)])
def test_lists_in_parts(m, cut, prec, masses):
    from oracle.pyoracle import Oracle
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.3, 0.2, 0.2), column=(0.3, 0.2, 0.2), dx=0.01, name="cells"))
    tb.scalars["nmaxpartj"] = cut or 5000
    g = tb.grid
    rng = np.random.default_rng(m)
    corner = g.extr_lo + g.dcd * np.array([4, 3, 3])
    # three cells a side; half of the particles in the middle one
    side = np.where(rng.random((m, 1)) < 0.5, rng.uniform(1.0, 2.0, (m, 3)), rng.uniform(0.0, 3.0, (m, 3)))
    far = g.extr_lo + g.dcd * (np.array([9, 6, 2]) + rng.uniform(0.05, 0.95, (40, 3)))
    coord = np.concatenate([corner + g.dcd * side, far])
    n = len(coord)
    dens = 1000.0 * (1.0 + rng.uniform(-1e-3, 1e-3, n))
    kw = dict(vel=rng.normal(0.0, 0.05, (n, 3)), dens=dens, pres=tb.case.bulk / 1000.0 * (dens - 1000.0),
              mass=np.where(np.arange(n) % masses == 0, 1e-5, 1.2e-5))
    o = Oracle(tb, coord=coord, semi=False, **kw)
    o.preloop()
    cnt_o, ids_o = o.lists()
    print(f"[gpu] m={m} cut={cut} prec={prec} masses={masses} longest list {cnt_o.max()}", flush=True)
    d = rt.SphContext(tb, precision=prec, capacity=n, semi=False)
    d.upload(coord=coord, **kw)
    d.preloop()
    p0 = d.pair_counter()
    cnt, ids = d.lists()
    assert np.array_equal(cnt, cnt_o) and p0 == cnt.sum() - n
    for i in range(n):
        assert np.array_equal(ids[i, :cnt[i]], ids_o[i, :cnt[i]]), i
    d.step(1)
    o.step(1)
    s, r = d.state(), o.state()
    d.close()
    for f in FIELDS:
        tol = 1e-4 * np.abs(r[f]).max() if prec else 0.0
        assert np.abs(s[f] - r[f]).max() <= tol, f
