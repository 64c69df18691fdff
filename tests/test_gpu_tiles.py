"""Tile forms of the pair passes.  A context's tile follows its capacity, so one
small solve is run in contexts of different capacity: every ladder entry, LDS
form and lane count.  A particle's sums do not depend on the tile (the list
order fixes them, and tiles that do not fit LDS use the same expressions), so
the states are equal bit for bit; the lists equal the oracle's, and the
smallest context is held to the oracle (FP64: equal; FP32-mixed: 1e-4 of each
field's largest value, the bar of the other FP32-mixed tests)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("coord", "vel", "acc", "dens", "pres", "dden", "vpres")


def _run(tb, coord, prec, capacity, steps, semi=True, **kw):
    from sphera_amd import runtime as rt
    d = rt.SphContext(tb, precision=prec, capacity=capacity, semi=semi)
    d.upload(coord=coord, **kw)
    d.preloop()
    lists = d.lists()
    d.step(steps)
    st = d.state()
    st["lists"], st["lists_end"] = lists, d.lists()
    d.close()
    return st


def _same(a, b):
    assert a["dt"] == b["dt"] and a["pairs"] == b["pairs"]
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), f
    for k in ("lists", "lists_end"):
        assert np.array_equal(a[k][0], b[k][0])
        for i in range(len(a[k][0])):
            n = a[k][0][i]
            assert np.array_equal(a[k][1][i, :n], b[k][1][i, :n])


def _oracle(tb, coord, steps, **kw):
    from oracle.pyoracle import Oracle
    o = Oracle(tb, coord=coord, **kw)
    o.preloop()
    lists = o.lists()
    o.step(steps)
    return o.state(), lists


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_every_tile_form(dim, prec):
    from sphera_amd import case2d
    from sphera_amd.case import DamBreak3D, build
    rng = np.random.default_rng(5)
    if dim == 3:
        tb = build(DamBreak3D(tank=(0.4, 0.2, 0.3), column=(0.12, 0.1, 0.12), dx=0.01, name="t"))
        caps = (1440, 8000, 14000, 25000, 38000, 50000, 80000, 120000, 300000)
    else:
        tb = case2d.build(case2d.DamBreak2D(tank=(0.6, 0.4), column=(0.3, 0.2), dx=0.01))
        caps = (600, 3000, 8000, 30000, 45000, 70000, 250000)
    c = tb.particles["coord"]
    j = rng.uniform(-0.1, 0.1, c.shape) * tb.case.dx
    if dim == 2:
        j[:, 1] = 0.0
    coord = c + j
    ref, lists = _oracle(tb, coord, 6)
    base = None
    for cap in caps:
        st = _run(tb, coord, prec, cap, 6)
        print(f"[gpu] dim={dim} prec={prec} capacity={cap}", flush=True)
        if base is None:
            base = st
            assert np.array_equal(st["lists"][0], lists[0])
            for i, n in enumerate(lists[0]):
                assert np.array_equal(st["lists"][1][i, :n], lists[1][i, :n])
            for f in FIELDS:
                tol = 1e-4 if prec == 1 else (1e-11 if dim == 2 else 0.0)  # 2D: the device's trigonometry
                assert np.abs(st[f] - ref[f]).max() <= tol * np.abs(ref[f]).max(), f
        else:
            _same(st, base)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("masses", [1, 2])
def test_tiles_beyond_lds(masses, prec):
    """A cluster far denser than water: its tiles exceed every LDS form in the
    small contexts, fit in others, and its lists are cut at NMAXPARTJ; one mass
    or two."""
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.2, 0.2, 0.2), column=(0.2, 0.2, 0.2), dx=0.01, name="cloud"))
    rng = np.random.default_rng(8)
    coord = np.concatenate([rng.uniform(0.085, 0.115, (2300, 3)), rng.uniform(0.03, 0.17, (900, 3))])
    n = len(coord)
    dens = 1000.0 * (1.0 + rng.uniform(-1e-3, 1e-3, n))
    kw = dict(vel=rng.normal(0.0, 0.05, (n, 3)), dens=dens,
              pres=tb.case.bulk / tb.case.rho0 * (dens - tb.case.rho0),
              mass=np.where(np.arange(n) % masses == 0, 1e-3, 1.2e-3))
    base = None
    for cap in (n, 14000, 50000, 120000, 300000):
        st = _run(tb, coord, prec, cap, 2, semi=False, **kw)
        print(f"[gpu] masses={masses} prec={prec} capacity={cap} longest list {st['lists'][0].max()}", flush=True)
        if base is None:
            base = st
            assert np.isfinite(st["acc"]).all()
        else:
            _same(st, base)
