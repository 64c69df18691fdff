"""The launch tunables of a case and its step time with them.

The kernels choose their launch shapes themselves (by capacity, h/dx and the
uploaded state), and the tunables of ``sph_params`` have no effect: there is
nothing to search, so ``autotune`` times a few steps of a scratch context and
returns the one ``tune`` dict, which ``SphContext`` accepts, with that time.

The grid's cell size is not a tunable: it is the reference's (CreaGrid), and
it fixes the neighbour-list order the device reproduces.
"""
from __future__ import annotations

import time


def _run(tb, coord, precision, tune, steps, warmup):
    from . import runtime as rt
    d = rt.SphContext(tb, precision=precision, tune=tune)
    try:
        d.upload(coord=coord)
        d.preloop()
        d.step(warmup)
        d.sync()
        t0 = time.perf_counter()
        d.step(steps)
        d.sync()
        return (time.perf_counter() - t0) / steps
    finally:
        d.close()


def autotune(tb, coord, precision, steps=4, warmup=2, log=None):
    """Returns (the tune dict, [(tune, seconds per step)])."""
    tune = dict(wg_size=64, chunk=8)
    s = _run(tb, coord, precision, tune, steps, warmup)
    if log:
        log(f"[autotune] precision={precision} {tune} -> {s * 1e3:.3f} ms/step")
    return tune, [(tune, s)]
