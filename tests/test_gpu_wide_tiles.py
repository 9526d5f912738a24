"""Levels small enough to run one 32x16 tile per compute unit, ragged sides
included, against 16x12 tiles."""
import numpy as np
import pytest

import ramses_amd as ra
from helpers import random_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sums", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,riemann,slope", [(56, "hll", 1), (64, "hllc", 1), (64, "exact", 8), (128, "llf", 2)])
def test_wide_tiles_same_bits(gpu, n, riemann, slope, precision, sums):
    from ramses_amd import autotune
    u = random_grid(np.random.default_rng(23), n, mach=2.0)
    ra.configure(gamma=1.4, riemann=riemann, slope_type=slope, precision=precision)
    out = []
    for tile in (5, 0, 4 if n % 32 == 0 else 0):
        autotune._set(autotune.LEVEL_TILE, tile)
        autotune._set(autotune.LEVEL_TZ, 0)
        lvl = ra.UniformLevel(u, sums=sums)
        lvl.step()
        lvl.step()
        out.append((lvl.u.cpu().numpy(), float(lvl.dt[0]), lvl.sums.cpu().numpy() if sums else None))
    autotune.reset()
    for v, dt, s in out[1:]:
        assert np.array_equal(v, out[0][0]) and dt == out[0][1]
        if sums:  # the same terms in another order
            np.testing.assert_allclose(s, out[0][2], rtol=n ** 3 * 2.3e-16)
    ra.configure()
