"""Neighbour lists at the edges of the search's 64-candidate chunks: one dense
cell of m particles (m around multiples of 64, and around the 640 candidates
the wavefront form holds), a second dense cell beside it, particles at exactly
2h, and a context with more capacity than particles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 127, 128, 129, 320, 576, 577, 639, 640, 641, 700])
def test_lists_at_chunk_edges(m):
    from oracle.pyoracle import Oracle
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.3, 0.2, 0.2), column=(0.3, 0.2, 0.2), dx=0.01, name="cell"))
    g = tb.grid
    rng = np.random.default_rng(m)
    corner = g.extr_lo + g.dcd * np.array([5, 4, 4])
    inside = corner + g.dcd * rng.uniform(0.02, 0.98, (m, 3))
    if m >= 2:  # a pair at 2h along x, to the last bit or beside it
        inside[1] = inside[0] + np.array([2.0 * tb.scalars["h"], 0.0, 0.0])
    far = g.extr_lo + g.dcd * (np.array([12, 9, 2]) + rng.uniform(0.05, 0.95, (3, 3)))
    coord = np.concatenate([inside, far])
    n = len(coord)
    kw = dict(vel=np.zeros((n, 3)), dens=np.full(n, 1000.0), pres=np.zeros(n), mass=np.full(n, 1e-3))
    o = Oracle(tb, coord=coord, **kw)
    o.preloop()
    cnt_o, ids_o = o.lists()
    print(f"[gpu] m={m} longest list {cnt_o.max()}", flush=True)
    d = rt.SphContext(tb, precision=rt.FP64, capacity=n + 77)
    d.upload(coord=coord, **kw)
    d.preloop()
    cnt, ids = d.lists()
    d.close()
    assert np.array_equal(cnt, cnt_o)
    for i in range(n):
        assert np.array_equal(ids[i, :cnt[i]], ids_o[i, :cnt[i]]), i
