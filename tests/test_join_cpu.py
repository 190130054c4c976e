"""Where the box join may stand in for the tree: without vertical edges the
oracle's tree finds exactly the pairs that brute force over all boxes finds,
also for rings on a small integer grid (shared x values, touching and
overlapping edges, one common largest x).  With vertical edges it does not,
which is why such rings stay with the tree."""
import numpy as np
import pytest

import oracle_py as O


def _grid_case(rng, vertical):
    """A base and one or two overlays on a small grid, with or without vertical edges."""
    while True:
        g = int(rng.integers(2, 9))
        b = rng.integers(0, g, (int(rng.integers(3, 9)), 2)).astype(float)
        cs = [rng.integers(0, g, (int(rng.integers(3, 9)), 2)).astype(float) + [float(rng.integers(-2, 4)), 0.0]
              for _ in range(int(rng.integers(1, 3)))]
        has = any(bool(np.any(r[:, 0] == np.roll(r[:, 0], -1))) for r in [b] + cs)
        if has == vertical:
            return b, cs


def _differs(b, cs):
    tr = O.Tree(b, cs)
    for k in range(1, len(cs) + 1):
        r = tr.clip(k, canonical=True)
        bb, bc, bt = tr.brute_pairs(k)
        if set(zip(r.pair_b, r.pair_c, r.pair_type)) != set(zip(bb, bc, bt)):
            return True
    return False


@pytest.mark.parametrize("seed", range(4))
def test_tree_equals_brute_force_without_vertical_edges(seed):
    rng = np.random.default_rng(seed)
    for _ in range(400):
        b, cs = _grid_case(rng, vertical=False)
        assert not _differs(b, cs), (b.tolist(), [c.tolist() for c in cs])


def test_tree_misses_pairs_with_vertical_edges():
    rng = np.random.default_rng(9)
    assert any(_differs(*_grid_case(rng, vertical=True)) for _ in range(200))
