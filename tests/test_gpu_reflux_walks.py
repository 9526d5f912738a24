"""The two ways to find the coarse leaves that a level's reflux corrects: from
the coarser level's cells and from the level's own sides.  A full coarser list
of more than 4096 octs behind a few fine ones takes the second, the part of it
around the fine octs alone the first: the same bits, and all of them conserve
mass, momenta and energy."""
import numpy as np
import pytest

import ramses_amd as ra
from amr_cases import smooth_state
from ramses_amd.tree import OctTree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [0.02, 0.06, 0.15])
@pytest.mark.parametrize("ivar,slope", [(0, 1), (1, 1), (0, 3)])
def test_reflux_walks(gpu, radius, ivar, slope):
    import torch
    from ramses_amd.amr import AmrLevels, configure_interpolation
    ball = lambda l, x: np.sqrt(((x - np.array([0.5, 0.46, 0.02])) ** 2).sum(1)) < radius  # noqa: E731
    tree = _tree(radius, ball)
    assert tree.n_octs(6) == 32768 and 6 * tree.n_octs(7) < 8 * 32768
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=slope)
    configure_interpolation(1, ivar)
    s = AmrLevels(tree, smooth_state(tree))
    pos = tree.grid_pos[tree.active[6]] + 0.5
    d = np.abs(pos / 32 - np.array([0.5, 0.46, 0.02]))
    near = tree.active[6][np.sqrt((np.minimum(d, 1 - d) ** 2).sum(1)) < radius + 0.12]
    assert len(near) <= 4096
    full, out = s.lists[6].clone(), []
    for part in (False, True):
        s.lists[6].copy_(full)
        s.nocts[6] = tree.n_octs(6)
        s.set_unew(6)
        s.set_unew(7)
        if part:
            s.lists[6][:len(near)] = torch.from_numpy(near.astype(np.int32)).cuda()
            s.nocts[6] = len(near)
        s.godunov(7, 2e-4)
        s.check()
        out.append(s.unew.clone())
    assert torch.equal(out[0], out[1])
    ngm, son = tree.ngridmax, np.concatenate([[0], tree.son])
    total = np.zeros((2, 5))
    for l, vol in ((6, 8.0), (7, 1.0)):
        c = (1 + np.arange(8)[:, None] * ngm + tree.active[l][None]).ravel()
        c = c[son[c] == 0]
        for k, u in enumerate((s.uold, out[0])):
            total[k] += vol * u.cpu().numpy()[:, c].sum(1)
    scale = np.abs(s.uold.cpu().numpy()).max() * 8 * 8 * 32768
    assert np.abs(total[1] - total[0]).max() < 1e-15 * scale
    changed = (out[0] != s.uold)[0].cpu().numpy()
    assert changed[(1 + np.arange(8)[:, None] * ngm + tree.active[6][None]).ravel()].sum() > 8
    ra.configure()


_trees = {}


def _tree(radius, ball):
    if radius not in _trees:
        _trees[radius] = OctTree(6, 7, ball)
    return _trees[radius]
