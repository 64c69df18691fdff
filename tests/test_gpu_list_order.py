"""Lists between a sort and the next search belong to the order before and are
not decoded: every count is 0; after the search they equal the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
def test_lists_between_sort_and_search(prec):
    from oracle.pyoracle import Oracle
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.3, 0.1, 0.2), column=(0.08, 0.1, 0.1), dx=0.01, name="t"))
    c = tb.particles["coord"]
    coord = c + np.random.default_rng(3).uniform(-0.05, 0.05, c.shape) * tb.case.dx
    o = Oracle(tb, coord=coord)
    d = rt.SphContext(tb, precision=prec)
    d.upload(coord=coord)
    assert not d.lists()[0].any()
    d.preloop()
    o.preloop()
    for ph in ("dt", "momentum", "velocity_smoothing", "sort"):
        assert np.array_equal(d.lists()[0], o.lists()[0]), ph
        d.phase(ph)
    assert not d.lists()[0].any()
    for ph in ("neighbours", "boundary_tab", "continuity", "pressure_smoothing"):
        d.phase(ph)
        assert d.lists()[0].all(), ph
    half = {k: v[: len(c) // 2] for k, v in tb.particles.items() if k in ("vel", "dens", "pres", "mass")}
    d.upload(coord=coord[: len(c) // 2], **half)  # a smaller solve in the same context
    cnt, _ = d.lists()
    assert len(cnt) == len(c) // 2 and not cnt.any()
    d.phase("neighbours")
    o = Oracle(tb, coord=coord[: len(c) // 2], **half)
    o.preloop()
    cnt, ids = d.lists()
    cnt_o, ids_o = o.lists()
    d.close()
    assert np.array_equal(cnt, cnt_o)
    for i, n in enumerate(cnt):
        assert np.array_equal(ids[i, :n], ids_o[i, :n])
