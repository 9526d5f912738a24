"""courant_fine with its conservation sums where the cells do not fill whole
workgroups, in a buffer of exactly the size asked for: numpy's sums, and not
a word behind the buffer."""
import ctypes

import numpy as np
import pytest

import ramses_amd as ra
from helpers import random_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 7, 8, 9, 10, 20, 30, 50, 101])
def test_courant_sums_stay_in_their_buffer(gpu, n):
    import torch
    ra.configure(gamma=1.4, riemann="hllc", slope_type=1, courant_factor=0.5)
    u = random_grid(np.random.default_rng(48), n, mach=1.0)
    d_u = torch.from_numpy(np.ascontiguousarray(u)).cuda()
    words = gpu.ramses_uniform_work_bytes(n) // 8
    work = torch.full((words + 64,), 7.0, dtype=torch.float64, device="cuda")
    dt, sums = (torch.zeros(k, dtype=torch.float64, device="cuda") for k in (1, 3))
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    rc = gpu.ramses_uniform_courant_sums(p(d_u), n, ctypes.c_double(1.0 / n), ctypes.c_double(1e10), p(dt), p(sums),
                                         p(work), ctypes.c_ulong(words * 8), None)
    torch.cuda.synchronize()
    assert rc == 0 and (work[words:] == 7.0).all()
    rho, m, e = u[0], u[1:4], u[4]
    ref = np.array([rho.sum(), e.sum(), (e - 0.5 * (m * m).sum(0) / rho).sum()]) / n ** 3
    np.testing.assert_allclose(sums.cpu().numpy(), ref, rtol=n ** 3 * 2.3e-16 + 1e-13)
    c = np.sqrt(1.4 * 0.4 * (e - 0.5 * (m * m).sum(0) / rho) / rho)
    k = (np.sqrt(1 + 2 * 0.5 * 1e-4) - 1) / 1e-4  # cmpdt without gravity (hydro/godunov_utils.f90:108-118)
    np.testing.assert_allclose(float(dt[0]), k / n / (3 * c + np.abs(m / rho).sum(0)).max(), rtol=1e-11)
    ra.configure()
