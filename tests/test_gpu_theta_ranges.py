"""FP64 parity with the CPU oracle for the generalised moncen slopes with a
theta far from 1: slopes down to the denormals reach the pressure terms'
divisions."""
import numpy as np
import pytest

import ramses_amd as ra
from helpers import NV, random_grid, random_stencils

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("riemann", ["hllc", "llf"])
@pytest.mark.parametrize("theta", [0.0, 1e-318, -1e-310, 1e-308, 3e-307, -1e-305, 1e-303, 1e-296, -1e-200, 2.0 ** -61, 2.0 ** -60, -900.0])
def test_theta_ranges(gpu, oracle_lib, theta, riemann):
    import torch
    rng = np.random.default_rng(50)
    k = dict(gamma=5 / 3, riemann=riemann, slope_type=8, slope_theta=theta)
    ra.configure(**k)
    oracle_lib.set_params(**k)
    u = random_stencils(rng, 8)
    f_ref, t_ref = np.zeros((8,) + ra.flux_shape(NV)), np.zeros((8,) + ra.tmp_shape(NV))
    # dt / dx of 1e307 lifts the traced states' terms of a slope of 1e-307
    for dt in (1e-4, 1e288, 1e305) if abs(theta) <= 1.0 else (1e-4,):  # MIN and MAX of a NaN are the compiler's choice
        oracle_lib.unsplit_batched(u, None, f_ref, t_ref, 0.01, dt)
        d_f = torch.zeros(f_ref.shape, dtype=torch.float64, device="cuda")
        d_t = torch.zeros(t_ref.shape, dtype=torch.float64, device="cuda")
        ra.unsplit_device(torch.from_numpy(u).cuda(), None, d_f, d_t, 0.01, dt)
        torch.cuda.synchronize()
        assert np.array_equal(d_f.cpu().numpy(), f_ref, equal_nan=True), dt
        assert np.array_equal(d_t.cpu().numpy(), t_ref, equal_nan=True), dt
    n = 24
    grid = random_grid(rng, n)
    lvl = ra.UniformLevel(grid)
    dt = float(lvl.step())
    ref, dt_ref = oracle_lib.uniform_step(grid, 1.0 / n)
    assert dt == dt_ref and np.array_equal(lvl.u.cpu().numpy(), ref, equal_nan=True)
    ra.configure()
