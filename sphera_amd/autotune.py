"""Launch-shape autotuner for the particle kernels.

The pair passes choose their workgroups by the solve's size (tiles of cells
held in LDS), so there is one shape left to time: for one case and precision a
scratch context runs a few steps, and the ``tune`` dict that ``SphContext`` /
``sph_params`` accept comes back with its time per step.

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
    """Returns (best tune dict, list of (tune, seconds per step))."""
    tune = dict(wg_size=64, chunk=8)
    s = _run(tb, coord, precision, tune, steps, warmup)
    if log:
        log(f"[autotune] precision={precision} {tune} -> {s * 1e3:.3f} ms/step")
    return tune, [(tune, s)]
