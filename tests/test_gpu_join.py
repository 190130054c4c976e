"""GPU checks of the box join that gives a clip its candidate pairs: the pairs,
rings and status of a clip against the staged tree calls (the general path) and
the oracle, at the edges of its leaves (64 edges) and groups (64 leaves), for
one pair, one base against many overlays and independent pairs; rings that it
must leave to the tree; and the tree's arrays and counts after a clip."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S
from fixtures import rings_equal, square, status_agrees
from test_join_cpu import _grid_case

pytestmark = pytest.mark.gpu

SIZES = [(3, 3), (63, 65), (64, 64), (65, 128), (129, 5), (7, 4096), (4096, 64), (4097, 4095), (9000, 300)]


def _tree_pairs(cl, ks):
    cl.reset()
    cl.build_tree().find_candidates()
    return [cl.pairs(k)[:2] for k in ks]


def _same_pairs(a, b):
    return all(np.array_equal(x, y) for p, q in zip(a, b) for x, y in zip(p, q))


@pytest.mark.parametrize("nb,nc", SIZES)
def test_pairs_at_leaf_and_group_edges(gpu, nb, nc):
    import segclip
    print("[gpu-join] star %d x %d" % (nb, nc), flush=True)
    b, c = S.star(nb, 31 + nb, 0.0, 0.0, 0.6, 1.0), S.star(nc, 77 + nc, 0.1, 0.05, 0.5, 1.0)
    cl = segclip.Clipper().set_polygons(b, [c])
    cl.clip(1)
    got, rings = cl.pairs(1), cl.rings()
    r = O.Tree(b, [c]).clip(1, canonical=True)
    assert np.array_equal(got[0], r.pair_b) and np.array_equal(got[1], r.pair_c) and np.array_equal(got[2], r.pair_type)
    assert rings_equal(rings, r.rings) is None
    assert _same_pairs([got[:2]], _tree_pairs(cl, [1]))


def test_one_base_many_overlays_and_three_levels(gpu):
    import segclip
    # a base of more than 64 groups (262,144 edges); overlays from one leaf up, one of them outside
    print("[gpu-join] harmonic 300,001 against ragged overlays", flush=True)
    b = S.harmonic(300001, 5)
    ovs = [S.star(n, 900 + n, 0.9 - 0.1 * i, 0.1 * i, 0.05, 0.3) for i, n in enumerate((3, 64, 65, 700, 4097, 20000))]
    ovs.append(S.star(40, 3, 50.0, 50.0, 0.5, 1.0))
    cl = segclip.Clipper().set_polygons(b, ovs)
    cl.clip_batch()
    ks = range(1, len(ovs) + 1)
    got = [cl.pairs(k)[:2] for k in ks]
    assert sum(len(p[0]) for p in got) > 100 and len(got[-1][0]) == 0
    assert _same_pairs(got, _tree_pairs(cl, ks))


def test_independent_pairs(gpu):
    import segclip
    bases, ovs = S.small_pairs(200, 4700)
    for n, m in SIZES:
        bases.append(S.star(n, 5 * n, 0.0, 0.0, 0.5, 1.0))
        ovs.append(S.star(m, 7 * m, 0.2, 0.1, 0.5, 1.0))
    print("[gpu-join] %d independent pairs" % len(bases), flush=True)
    cl = segclip.Clipper().set_pairs(bases, ovs)
    cl.clip_batch()
    ks = range(1, len(bases) + 1)
    got = [cl.pairs(k)[:2] for k in ks]
    assert _same_pairs(got, _tree_pairs(cl, ks))


@pytest.mark.parametrize("vertical", [False, True])
def test_grid_rings_equal_the_oracle(gpu, vertical):
    import segclip
    rng = np.random.default_rng(12)
    for i in range(60):
        b, cs = _grid_case(rng, vertical)
        print("[gpu-join] grid %d" % i, flush=True)
        tr = O.Tree(b, cs)
        cl = segclip.Clipper().set_polygons(b, cs)
        for k in range(1, len(cs) + 1):
            cl.clip(k)
            r = tr.clip(k, canonical=True)
            p = cl.pairs(k)
            assert np.array_equal(p[0], r.pair_b) and np.array_equal(p[1], r.pair_c) and np.array_equal(p[2], r.pair_type)
            assert status_agrees(int(cl.batch_status()[0]), r.status)
        cl.close()


def test_tree_arrays_and_counts_after_a_clip(gpu):
    import segclip
    b, ovs = S.star1k()
    ref = segclip.Clipper().set_polygons(b, ovs)
    ref.build_tree().find_candidates()
    want, wc = [ref.elementary(), ref.node_intervals()[2:], ref.cover_lists()[0], ref.leaf_targets()[0]], ref.counts()
    for first in range(2):
        cl = segclip.Clipper().set_polygons(b, ovs)
        cl.clip(1)
        rings = cl.rings()
        if first:  # the counts first, then the arrays; and the other way round
            gc = cl.counts()
        got = [cl.elementary(), cl.node_intervals()[2:], cl.cover_lists()[0], cl.leaf_targets()[0]]
        gc = cl.counts()
        for g, w in zip(got, want):
            assert np.array_equal(g, w)
        for k in ("epc", "tree_size", "cover_entries", "leaf_end_entries", "tests", "candidates", "pairs", "stab_units",
                  "near_pairs"):
            assert gc[k] == wc[k], k
        assert rings_equal(cl.rings(), rings) is None
        cl.materialize_end_lists()
        assert len(cl.end_lists()[1]) > 0


def test_squares_keep_the_tree(gpu):
    import segclip
    cl = segclip.Clipper().set_polygons(square(2.0, 3.0, 3.0, 4.0), [square(2.0, 1.0, 4.0, 6.0)])
    cl.clip(1)
    r = O.Tree(square(2.0, 3.0, 3.0, 4.0), [square(2.0, 1.0, 4.0, 6.0)]).clip(1, canonical=True)
    p = cl.pairs(1)
    assert np.array_equal(p[0], r.pair_b) and np.array_equal(p[1], r.pair_c)
