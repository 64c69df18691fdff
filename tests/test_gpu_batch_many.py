"""Batches of many small solves with walls: every segment equals the same solve
alone, bit for bit (segments of different spacing, so of different wall
tables, some of them without the ring structure; more key blocks than segments and more segments than a workgroup's key
blocks)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("coord", "vel", "acc", "dens", "pres", "dden", "vpres")


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("count", [3, 40])
def test_segments_equal_single_solves(count, prec):
    from sphera_amd import runtime as rt
    from sphera_amd.case import DamBreak3D, build
    tbs = [build(DamBreak3D(tank=(0.3, 0.12, 0.2), column=(0.06 + 0.01 * (k % 4), 0.12, 0.06 + 0.013 * (k % 5)),
                            dx=0.01 + 0.0007 * (k % 3), name=f"s{k}")) for k in range(min(count, 12))]
    for tb in tbs[1::3]:
        tb.bitab = tb.bitab.copy()
        tb.bitab[37, 3] *= 1.0 + 1.0e-7
    tbs = [tbs[k % 12] for k in range(count)]
    rng = np.random.default_rng(2)
    coords = [tb.particles["coord"] + rng.uniform(-0.2, 0.2, tb.particles["coord"].shape) * tb.case.dx for tb in tbs]
    print(f"[gpu] {count} segments prec={prec}", flush=True)
    b = rt.SphBatch(tbs, precision=prec)
    b.upload(coords=coords)
    b.preloop()
    b.step(4)
    for k, (tb, x) in enumerate(zip(tbs, coords)):
        d = rt.SphContext(tb, precision=prec)
        d.upload(coord=x)
        d.preloop()
        d.step(4)
        s, g = d.state(), b.seg_state(k)
        d.close()
        assert s["dt"] == g["dt"]
        for f in FIELDS:
            assert np.array_equal(s[f], g[f]), (k, f)
    b.close()
