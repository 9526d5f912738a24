"""The refinement map and the rebuilt grid lists against a few lines of numpy,
at sizes that span several workgroups and scan tiles and leave remainders."""
import numpy as np
import pytest

import ramses_amd as ra
from ramses_amd.tree import OctTree

pytestmark = pytest.mark.gpu


def _mesh(tree, nlevelmax):
    from ramses_amd.amr import AmrLevels, configure_interpolation, configure_refinement
    ra.configure(gamma=5 / 3, riemann="hllc", slope_type=1)
    configure_interpolation(1, 0)
    configure_refinement()
    u = np.ones((5, tree.ncell))
    return AmrLevels(tree, u, nlevelmax=nlevelmax)


def _smooth(flag, exist):
    """smooth_fine's three passes on a periodic lattice."""
    for nthr in (1, 2, 2):
        n = sum(np.roll(flag, s, a) for a in range(3) for s in (1, -1))
        flag = ((flag == 1) | (n >= nthr)).astype(int) * exist
    return flag


@pytest.mark.parametrize("nexpand", [0, 1, 2])
@pytest.mark.parametrize("radius", [None, 0.33])
@pytest.mark.parametrize("level", [3, 5])
def test_flag_smoothing(gpu, level, radius, nexpand):
    """flag_fine without criteria: random flags of the next level's cells, on
    a full level and on one with an edge, smoothed 1 + nexpand times."""
    import torch
    from ramses_amd.amr import configure_refinement
    rng = np.random.default_rng(41)
    if radius is None:  # the map of a full level
        lmin, l = level, level
        tree = OctTree(level, level + 1, lambda k, x: rng.random(len(x)) < 0.1, nexpand=0)
    else:
        lmin, l = level - 1, level
        inside = lambda k, x: np.sqrt(((x - 0.5) ** 2).sum(1)) < radius * 0.5 ** (k - lmin)  # noqa: E731
        tree = OctTree(lmin, level + 1, inside)
    s = _mesh(tree, level + 2)
    configure_refinement(nexpand=nexpand)
    n = 2 ** l
    flag1 = np.zeros(tree.ncell + 1, dtype=np.int32)
    ci, cx = tree.cells_of_level(l + 1)
    flag1[ci] = rng.random(len(ci)) < 0.05
    s.flag1.copy_(torch.from_numpy(flag1))
    s.flag(l, 2, lmin)  # icount 2: no ensure_ref_rules
    ic, x = tree.cells_of_level(l)
    at = tuple((x[:, a] * n).astype(int) for a in (2, 1, 0))
    exist, flag = np.zeros((n, n, n), dtype=int), np.zeros((n, n, n), dtype=int)
    exist[at] = 1
    son = np.concatenate([[0], tree.son])
    kids = son[ic]
    ngm = tree.ngridmax
    init = np.zeros(len(ic), dtype=int)
    for k in range(8):
        cc = 1 + k * ngm + kids
        init |= (kids > 0) & ((son[np.where(kids > 0, cc, 0)] > 0) | (flag1[np.where(kids > 0, cc, 0)] == 1))
    flag[at] = init
    assert init.any() and not init.all()
    for _ in range(1 + nexpand):
        flag = _smooth(flag, exist)
    assert np.array_equal(s.flag1.cpu().numpy()[ic], flag[at])
    configure_refinement()


@pytest.mark.parametrize("level,share", [(3, 0.3), (5, 0.02), (5, 0.5)])
def test_refine_order(gpu, level, share):
    """refine_fine of a full level from random maps, twice: the new octs take
    the free grids in the order in which nvector batches visit the cells, the
    killed ones go behind them, and the list is survivors, then new octs."""
    import torch
    rng = np.random.default_rng(42)
    tree = OctTree(level, level, extra_grids=2 * 8 ** level)
    s = _mesh(tree, level + 1)
    ngm, noct = tree.ngridmax, 8 ** (level - 1)
    active = np.asarray(tree.active[level])
    batches = [active[b:b + 32] for b in range(0, noct, 32)]
    order = np.concatenate([1 + ind * ngm + b for b in batches for ind in range(8)])  # the visit order of the cells
    free, grids = list(s.free_list()), []
    son = {}
    for _ in range(2):
        want = rng.random(len(order)) < share
        flag1 = s.flag1.cpu().numpy()
        flag1[order] = want
        s.flag1.copy_(torch.from_numpy(flag1))
        make = [c for c, w in zip(order, want) if w and c not in son]
        kill = [c for c, w in zip(order, want) if not w and c in son]
        new, free = free[:len(make)], free[len(make):]
        dead = [son.pop(c) for c in kill]
        grids = [g for g in grids if g not in set(dead)] + new
        free += dead
        son.update(zip(make, new))
        s.refine(level)
        s.check()
        assert s.noct(level + 1) == len(grids) and np.array_equal(s.grids(level + 1), grids)
        assert np.array_equal(s.free_list(), free)
        got = s.son.cpu().numpy()
        assert all(got[c] == son.get(c, 0) for c in order)
        assert np.array_equal(s.pos.cpu().numpy()[grids], np.arange(len(grids)))
