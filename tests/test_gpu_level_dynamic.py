"""Levels with the solvers that are not fixed at compile time, in FP32-mixed:
the chunk rule and the update of their own (the conserved state loaded again
with minmod, kept with the others) against 8x8 tiles in chunks of 4, and
close to the FP64 step."""
import numpy as np
import pytest

import ramses_amd as ra
from helpers import random_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sums", [False, True])
@pytest.mark.parametrize("slope", [1, 2])
@pytest.mark.parametrize("riemann", ["acoustic", "exact"])
@pytest.mark.parametrize("n", [8, 40, 72, 176])
def test_dynamic_solver_levels(gpu, n, riemann, slope, sums):
    from ramses_amd import autotune
    u = random_grid(np.random.default_rng(49), n, mach=0.5)
    out = []
    for precision, tile, tz in (("fp32", 3, 4), ("fp32", 0, 0), ("fp64", 0, 0)):
        ra.configure(gamma=1.4, riemann=riemann, slope_type=slope, precision=precision)
        autotune._set(autotune.LEVEL_TILE, tile)
        autotune._set(autotune.LEVEL_TZ, tz)
        lvl = ra.UniformLevel(u, sums=sums)
        lvl.step()
        out.append((lvl.u.cpu().numpy(), float(lvl.dt[0]), lvl.sums.cpu().numpy() if sums else None))
    autotune.reset()
    ra.configure()
    (a, dt, s), (b, dt2, s2), (c, _, s3) = out
    assert np.array_equal(a, b) and dt == dt2
    assert np.abs(a - c).max() < 1e-4 * np.abs(c).max()
    if sums:
        np.testing.assert_allclose(s2, s, rtol=n ** 3 * 2.3e-16)
        np.testing.assert_allclose(s2, s3, rtol=1e-6)
