"""2D corner quadratures, one point a lane: more corner particles in a
workgroup than its lane groups take at once, at the tolerance of the 2D
boundary tables."""
import numpy as np
import pytest

from sphera_amd import case2d
from tests.test_gpu_2d import SMALL, _btab_close, _jitter2d, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 9, 17, 33])
def test_corner_tables_match_oracle(n):
    tb = case2d.build(case2d.DamBreak2D(**SMALL))
    dx = tb.case.dx
    coord = _jitter2d(tb.particles["coord"], dx)
    rng = np.random.default_rng(n)
    pick = rng.choice(len(coord), n, replace=False)
    for d in (0, 2):
        coord[pick, d] = coord[:, d].min() + rng.uniform(0.0, 2.2, n) * dx
    d, o = _pair(tb, 0, coord)
    assert _btab_close(d, o) >= 2 * n
    d.close()
