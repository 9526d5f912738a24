"""A direct coarse step in a workspace of the caller's: no library state, no
allocation, so that a program can also capture it; whatever the buffer held
before."""
import numpy as np
import pytest

import ramses_amd as ra
from amr_cases import smooth_state, sphere_tree

pytestmark = pytest.mark.gpu


def _solver(sums, own):
    import torch
    from ramses_amd.amr import AmrSolver, configure_interpolation
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=1)
    configure_interpolation(1, 0)
    tree = sphere_tree(levelmin=3, levelmax=5)
    s = AmrSolver(tree, smooth_state(tree), sums=sums)
    buf = None
    if own:
        # exactly what the largest level asks for, full of ones
        need = max(s.lib.ramses_amr_work_bytes(s.noct(l)) for l in range(1, 6))
        buf = torch.full((need,), 255, dtype=torch.uint8, device="cuda")
        s._mesh.work, s._mesh.work_bytes = buf.data_ptr(), need
    return s, buf


def _state(s):
    return [getattr(s, a).clone() for a in ("uold", "dt", "dtold", "time")] + ([] if s.sums is None else [s.sums.clone()])


@pytest.mark.parametrize("sums", [False, True])
def test_own_workspace(gpu, sums):
    import torch
    ref, _ = _solver(sums, False)
    s, buf = _solver(sums, True)
    try:
        for _ in range(3):
            ref.coarse_step()
            s.coarse_step()
            assert s._mesh.work == buf.data_ptr() and not s._mesh.graph_state and not ref._mesh.graph_state
            assert all(torch.equal(a, b) for a, b in zip(_state(ref), _state(s)))
            buf.fill_(255)  # the caller's between steps
    finally:
        s._mesh.work, s._mesh.work_bytes = None, 0


def test_first_step_captured(gpu):
    import torch
    ref, _ = _solver(True, False)
    s, buf = _solver(True, True)
    try:
        s.nstep_coarse_old = -1  # the baselines are a later step's
        ref.nstep_coarse_old = -1
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            s.coarse_step()
        for _ in range(4):
            ref.coarse_step()
            g.replay()
            buf.fill_(255)
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(_state(ref), _state(s)))
    finally:
        s._mesh.work, s._mesh.work_bytes = None, 0
