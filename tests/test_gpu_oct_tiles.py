"""The 16-oct tiles of the batched unsplit and of the oct-tree level sweep
where they are ragged: fewer octs than a tile, one more, tiles that span
batches, a short last batch.  Bitwise against the CPU oracle in FP64."""
import numpy as np
import pytest

import ramses_amd as ra
from helpers import conserved, random_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gravity", [False, True])
@pytest.mark.parametrize("nv,groups,last", [(32, 1, 1), (32, 1, 15), (32, 1, 16), (32, 1, 17), (32, 2, 0), (32, 3, 31),
                                            (1, 1, 1), (1, 17, 1), (7, 5, 3), (16, 2, 16), (24, 3, 9), (37, 2, 36)])
def test_unsplit_ragged_tiles(gpu, oracle_lib, nv, groups, last, gravity):
    import torch
    rng = np.random.default_rng(11)
    shape = (groups, 6, 6, 6, nv)
    u = np.ascontiguousarray(np.moveaxis(conserved(rng.lognormal(0.0, 1.0, shape), rng.normal(0.0, 1.0, (3,) + shape),
                                                   rng.lognormal(-0.5, 0.5, shape), 5 / 3), 0, 1))
    g = rng.normal(0.0, 1.0, (groups,) + ra.grav_shape(nv)) if gravity else None
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=1, nvector=nv)
    oracle_lib.set_params(gamma=5 / 3, riemann="hllc", slope_type=1)
    f_ref, t_ref = np.full((groups,) + ra.flux_shape(nv), 3.0), np.full((groups,) + ra.tmp_shape(nv), 3.0)
    oracle_lib.unsplit_batched(u, g, f_ref, t_ref, 0.01, 1e-4, ngrid_last=last)
    d_f, d_t = (torch.full(r.shape, 3.0, dtype=torch.float64, device="cuda") for r in (f_ref, t_ref))
    ra.unsplit_device(torch.from_numpy(u).cuda(), None if g is None else torch.from_numpy(g).cuda(), d_f, d_t, 0.01,
                      1e-4, ngrid_last=last)
    torch.cuda.synchronize()
    assert np.array_equal(d_f.cpu().numpy(), f_ref) and np.array_equal(d_t.cpu().numpy(), t_ref)
    ra.configure()


@pytest.mark.parametrize("riemann,slope", [("hllc", 1), ("llf", 2)])
@pytest.mark.parametrize("level,octs", [(3, 64), (4, 512), (4, 1), (4, 16), (4, 17), (4, 495)])
def test_level_sweep_ragged_tiles(gpu, oracle_lib, level, octs, riemann, slope):
    """godunov_fine of a full level, or of the first `octs` octs of its list:
    the update of their cells is the uniform level's, the others keep unew."""
    from ramses_amd.amr import AmrLevels, configure_interpolation
    from ramses_amd.tree import OctTree
    rng = np.random.default_rng(12)
    n = 2 ** level
    tree = OctTree(level, level)
    grid = random_grid(rng, n)
    cells, x = tree.cells_of_level(level)
    at = tuple((x[:, a] * n).astype(int) for a in (2, 1, 0))
    u = np.ones((5, tree.ncell))
    u[:, cells - 1] = grid[(slice(None),) + at]
    ra.configure(gamma=5 / 3, riemann=riemann, slope_type=slope)
    oracle_lib.set_params(gamma=5 / 3, riemann=riemann, slope_type=slope)
    configure_interpolation(1, 0)
    s = AmrLevels(tree, u)
    s.set_unew(level)
    s.nocts[level] = octs
    s.godunov(level, 1e-3)
    s.check()
    ref = oracle_lib.uniform_godunov(grid, 1.0 / n, 1e-3)
    swept = np.isin((cells - 2) % tree.ngridmax + 1, tree.active[level][:octs])
    want = np.where(swept, ref[(slice(None),) + at], grid[(slice(None),) + at])
    assert np.array_equal(s.state("new")[:, cells - 1], want)
    ra.configure()
