"""Level tiles and z chunks that reach past the level: sides that no tile
divides, the smallest sides, several sizes in one batched launch."""
import numpy as np
import pytest

import ramses_amd as ra
from helpers import random_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sums", [False, True])
@pytest.mark.parametrize("n", [8, 16, 24, 32, 40, 56, 72, 88])
def test_ragged_level_vs_oracle(gpu, oracle_lib, n, sums):
    rng = np.random.default_rng(21)
    u = random_grid(rng, n, mach=2.0)
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=1, courant_factor=0.5)
    oracle_lib.set_params(gamma=5 / 3, riemann="hllc", slope_type=1, courant_factor=0.5)
    lvl = ra.UniformLevel(u, sums=sums)
    dt = float(lvl.step())
    ref, dt_ref = oracle_lib.uniform_step(u, 1.0 / n)
    assert dt == dt_ref and np.array_equal(lvl.u.cpu().numpy(), ref)
    dt2, mass, e, eint = oracle_lib.uniform_courant(ref, 1.0 / n, 1.0 / 1e-10)
    assert float(lvl.dt[0]) == dt2
    if sums:  # n^3 terms, each once: the order alone differs
        np.testing.assert_allclose(lvl.sums.cpu().numpy(), [mass, e, eint], rtol=n ** 3 * 2.3e-16)
    ra.configure()


@pytest.mark.parametrize("n", [24, 40, 64, 88])
def test_ragged_level_fp32_same_bits_on_every_tile(gpu, n):
    """FP32-mixed: 8x8 tiles, which divide every side, against the default."""
    from ramses_amd import autotune
    u = random_grid(np.random.default_rng(22), n, mach=2.0)
    ra.configure(gamma=5 / 3, riemann="llf", slope_type=2, precision="fp32")
    out = []
    for tile, tz in ((3, 4), (0, 0), (5, 8)):
        autotune._set(autotune.LEVEL_TILE, tile)
        autotune._set(autotune.LEVEL_TZ, tz)
        lvl = ra.UniformLevel(u)
        lvl.step()
        out.append((lvl.u.cpu().numpy(), float(lvl.dt[0])))
    autotune.reset()
    for v, dt in out[1:]:
        assert np.array_equal(v, out[0][0]) and dt == out[0][1]
    ra.configure()


def test_batched_sizes_same_bits_as_alone(gpu):
    """Slots of sides that no 16x12 tile divides advance together and alone to
    the same bits, FP64, the last step of each shortened to its end time."""
    import torch
    from ramses_amd.serve import HydroServer, Request
    sides = [16, 32, 48, 16, 80]
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=1, courant_factor=0.5)
    ics = [torch.from_numpy(random_grid(np.random.default_rng(30 + i), n)).cuda() for i, n in enumerate(sides)]

    def serve(ids):
        reqs = [Request(i, sides[i], 2e-3, ic=lambda n, i=i: ics[i], keep_result=True) for i in ids]
        HydroServer().run(reqs)
        return {r.id: (r.steps, r.result.cpu().numpy()) for r in reqs}
    together = serve(range(len(sides)))
    for i in range(len(sides)):
        steps, u = serve([i])[i]
        assert steps == together[i][0] >= 1 and np.array_equal(u, together[i][1])
    ra.configure()
