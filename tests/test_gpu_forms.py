"""Forms of the pair passes: on tiles in LDS, or gathering for every particle
(clusters whose tiles do not fit, thin clouds, FP64 with several masses, tiles of
one cell, FP64 tiles that fill their last round badly).  Against the oracle: FP64 equal,
FP32-mixed within 1e-4 of each field's largest value, the bar of the other
tests; between contexts that take different forms, lane counts and batches: bit
for bit; captured steps are not replayed in another form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("coord", "vel", "acc", "dens", "pres", "dden", "vpres")


def _cluster(masses, n0=2300, n1=900, **kw):
    """A cluster far denser than water in a thin cloud."""
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.2, 0.2, 0.2), column=(0.2, 0.2, 0.2), dx=0.01, name="cloud", **kw))
    rng = np.random.default_rng(8)
    coord = np.concatenate([rng.uniform(0.085, 0.115, (n0, 3)), rng.uniform(0.03, 0.17, (n1, 3))])
    n = len(coord)
    dens = 1000.0 * (1.0 + rng.uniform(-1e-3, 1e-3, n))
    st = dict(coord=coord, vel=rng.normal(0.0, 0.05, (n, 3)), dens=dens,
              pres=tb.case.bulk / tb.case.rho0 * (dens - tb.case.rho0),
              mass=np.where(np.arange(n) % masses == 0, 1e-3, 1.2e-3) / 20.0)
    return tb, st


def _water(dx=0.01, trunc=1.3, column=(0.12, 0.1, 0.12), masses=1, **kw):
    from sphera_amd.case import DamBreak3D, build
    tb = build(DamBreak3D(tank=(0.4, 0.2, 0.3), column=column, dx=dx, trunc=trunc, name="w", **kw))
    P = tb.particles
    rng = np.random.default_rng(5)
    st = {k: P[k].copy() for k in ("coord", "vel", "dens", "pres", "mass")}
    st["coord"] += rng.uniform(-0.1, 0.1, P["coord"].shape) * dx
    st["mass"] *= np.where(np.arange(len(P["mass"])) % masses == 0, 1.0, 1.1)
    return tb, st


def _run(tb, st, prec, steps, capacity=None, semi=True):
    from sphera_amd import runtime as rt
    d = rt.SphContext(tb, precision=prec, capacity=capacity or len(st["coord"]), semi=semi)
    d.upload(**st)
    d.preloop()
    d.step(steps)
    s = d.state()
    s["lists"] = d.lists()
    d.close()
    return s


def _held(s, r, prec):
    for f in FIELDS:
        tol = 1e-4 * np.abs(r[f]).max() if prec else 0.0
        assert np.abs(s[f] - r[f]).max() <= tol, f


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("masses", [1, 2])
@pytest.mark.parametrize("n1", [900, 12000])  # most particles in tiles that do not fit, few
def test_clusters_match_oracle(n1, masses, prec):
    from oracle.pyoracle import Oracle
    tb, st = _cluster(masses, n1=n1)
    o = Oracle(tb, semi=False, **st)
    o.preloop()
    o.step(2)
    cnt, ids = o.lists()
    print(f"[gpu] cluster {n1} masses={masses} prec={prec} longest list {cnt.max()}", flush=True)
    for capacity in (None, 50000, 300000):
        s = _run(tb, st, prec, 2, capacity, semi=False)
        assert np.array_equal(s["lists"][0], cnt)
        for i, k in enumerate(cnt):
            assert np.array_equal(s["lists"][1][i, :k], ids[i, :k]), i
        _held(s, o.state(), prec)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("rk1", [False, True])
@pytest.mark.parametrize("trunc,masses", [(1.3, 1), (1.3, 2), (2.0, 1), (2.0, 2)])
def test_water_matches_oracle(trunc, masses, rk1, prec):
    from oracle.pyoracle import Oracle
    tb, st = _water(trunc=trunc, masses=masses, time_split=0 if rk1 else 1)
    o = Oracle(tb, **st)
    o.preloop()
    o.step(4)
    base = None
    for capacity in (None, 25000, 80000, 300000):
        print(f"[gpu] trunc={trunc} masses={masses} rk1={rk1} prec={prec} capacity={capacity}", flush=True)
        s = _run(tb, st, prec, 4, capacity)
        if base is None:
            base = s
            _held(s, o.state(), prec)
        for f in FIELDS:
            assert np.array_equal(s[f], base[f]), f


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind", ["clusters", "masses", "half"])
def test_batches_gather(kind, prec):
    """Segments equal their own contexts' results: all of them gathering, or one
    of two."""
    from sphera_amd import runtime as rt
    cases = {"clusters": [_cluster(1), _cluster(1, n0=1700, n1=333)], "masses": [_water(masses=2), _water(dx=0.0113, masses=2)],
             "half": [_water(column=(0.3, 0.2, 0.2)), _cluster(1, n0=400, n1=31)]}[kind]
    for tb, st in cases:
        tb.particles.update(st)
    semi = kind == "masses"
    b = rt.SphBatch([tb for tb, _ in cases], precision=prec, semi=semi)
    b.upload()
    b.preloop()
    b.step(2)
    b.step_graph(1)
    b.sync()
    for k, (tb, st) in enumerate(cases):
        print(f"[gpu] batch {kind} prec={prec} segment {k}", flush=True)
        s, g = _run(tb, st, prec, 3, semi=semi), b.seg_state(k)
        for f in FIELDS:
            assert np.array_equal(s[f], g[f]), f
    b.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_form_changes_between_uploads(prec):
    from sphera_amd import runtime as rt
    tb, dense = _cluster(1)
    thin = {k: v[-900:] for k, v in dense.items()}
    two = dict(thin, mass=thin["mass"] * np.where(np.arange(900) % 2 == 0, 1.0, 1.1))
    d = rt.SphContext(tb, precision=prec, capacity=3200, semi=False)
    for st in (thin, dense, two, thin, dense):
        d.upload(**st)
        d.preloop()
        for _ in range(3):
            d.step_graph(1)
        d.sync()
        s, r = d.state(), _run(tb, st, prec, 3, 3200, semi=False)
        for f in FIELDS:
            assert np.array_equal(s[f], r[f]), f
    d.close()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind", ["gathers", "tiles"])
@pytest.mark.parametrize("cut", [1, 8, 9, 16])
def test_short_lists(cut, kind, prec):
    """Lists cut at NMAXPARTJ of less than two groups of entries."""
    from oracle.pyoracle import Oracle
    tb, st = _cluster(1, n0=500, n1=300) if kind == "gathers" else _water(column=(0.3, 0.2, 0.2))
    tb.scalars["nmaxpartj"] = cut
    print(f"[gpu] cut={cut} {kind} prec={prec}", flush=True)
    o = Oracle(tb, semi=False, **st)
    o.preloop()
    o.step(1)
    s = _run(tb, st, prec, 1, semi=False)
    _held(s, o.state(), prec)
    cnt, ids = o.lists()
    assert np.array_equal(s["lists"][0], cnt)
    for i, k in enumerate(cnt):
        assert np.array_equal(s["lists"][1][i, :k], ids[i, :k]), i
