"""FP64 parity with the CPU oracle where divisions leave the range of the
shared reciprocals: values from far below to far above it, alone and mixed
into the same wavefronts, and parameters that switch the range off.  The
wide values reach 0/0 in some faces: NaN equals NaN there."""
import numpy as np
import pytest

import ramses_amd as ra
from helpers import NV, conserved

pytestmark = pytest.mark.gpu


def _primitives(rng, mode, shape):
    sign = rng.choice([-1.0, 1.0], (3,) + shape)
    if mode == "wide":  # both sides of every bound, zero velocities among them
        rho = 10 ** rng.uniform(-13, 20, shape)
        vel = sign * 10 ** rng.uniform(-330, 25, (3,) + shape) * (rng.random((3,) + shape) > 0.2)
        return rho, vel, 10 ** rng.uniform(-60, 20, shape)
    if mode == "quiet":  # a uniform gas, velocities down to the denormals
        vel = sign * 10 ** rng.uniform(-322, -10, (3,) + shape) * (rng.random((3,) + shape) > 0.5)
        return np.ones(shape), vel, np.full(shape, 1e-5)
    rho = rng.lognormal(0.0, 1.0, shape)  # "edge": ordinary, a few cells far outside
    odd = rng.random(shape) < 0.01
    return (np.where(odd, 1e17, rho), sign * rng.lognormal(0.0, 1.0, (3,) + shape),
            np.where(rng.random(shape) < 0.01, 1e18, rng.lognormal(-0.5, 0.5, shape)))


@pytest.mark.parametrize("smallr", [1e-10, 1e-25])
@pytest.mark.parametrize("mode", ["wide", "quiet", "edge"])
@pytest.mark.parametrize("riemann,slope", [("hllc", 1), ("hllc", 2), ("hll", 1), ("hll", 8), ("llf", 7)])
def test_unsplit_division_ranges(gpu, oracle_lib, riemann, slope, mode, smallr):
    rng = np.random.default_rng(5)
    G = 6
    u = np.ascontiguousarray(np.moveaxis(conserved(*_primitives(rng, mode, (G, 6, 6, 6, NV)), 5 / 3), 0, 1))
    ra.configure(gamma=5 / 3, riemann=riemann, slope_type=slope, smallr=smallr)
    oracle_lib.set_params(gamma=5 / 3, riemann=riemann, slope_type=slope, smallr=smallr)
    import torch
    d_u = torch.from_numpy(u).cuda()
    for dx in (1 / 64, 0.01):  # a power of two, and one whose division is a division
        f_ref, t_ref = np.zeros((G,) + ra.flux_shape(NV)), np.zeros((G,) + ra.tmp_shape(NV))
        oracle_lib.unsplit_batched(u, None, f_ref, t_ref, dx, 1e-4)
        d_f = torch.zeros(f_ref.shape, dtype=torch.float64, device="cuda")
        d_t = torch.zeros(t_ref.shape, dtype=torch.float64, device="cuda")
        ra.unsplit_device(d_u, None, d_f, d_t, dx, 1e-4)
        torch.cuda.synchronize()
        assert np.array_equal(d_f.cpu().numpy(), f_ref, equal_nan=True), dx
        assert np.array_equal(d_t.cpu().numpy(), t_ref, equal_nan=True), dx
    ra.configure()


@pytest.mark.parametrize("mode", ["wide", "quiet", "edge"])
@pytest.mark.parametrize("n", [16, 24, 48])
def test_level_division_ranges(gpu, oracle_lib, n, mode):
    rng = np.random.default_rng(6)
    u = np.ascontiguousarray(conserved(*_primitives(rng, mode, (n, n, n)), 5 / 3))
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=1, courant_factor=0.5)
    oracle_lib.set_params(gamma=5 / 3, riemann="hllc", slope_type=1, courant_factor=0.5)
    lvl = ra.UniformLevel(u)
    dt = float(lvl.step())
    ref, dt_ref = oracle_lib.uniform_step(u, 1.0 / n)
    assert dt == dt_ref and np.array_equal(lvl.u.cpu().numpy(), ref, equal_nan=True)
    if np.isfinite(ref).all():  # MIN and MAX of a NaN are the compiler's choice
        assert float(lvl.dt[0]) == oracle_lib.uniform_courant(ref, 1.0 / n, 1.0 / 1e-10)[0]
    ra.configure()
