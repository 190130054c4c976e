"""GPU checks of a clip after some of the tree's stages: the candidates come from
the join, and the calls that show the tree or its counts have to find all of it
built, not only the stages that were called."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S
from fixtures import rings_equal, square

pytestmark = pytest.mark.gpu

STAGES = ["elementary", "node_intervals", "end_lists", "cover_lists"]


def _call(cl, name):
    import segclip
    cl._check(getattr(segclip.lib(), "segclip_build_" + name)(cl._h))


def _tree(cl):
    off, e = cl.cover_lists()
    return [cl.elementary(), cl.node_intervals(), off, np.sort(e), cl.leaf_targets()[0], cl.leaf_targets()[1]]


@pytest.mark.parametrize("stages", [1, 2, 3, 4])
@pytest.mark.parametrize("again", [False, True])
def test_clip_after_some_stages(gpu, stages, again):
    import segclip
    b, ovs = S.star1k()
    ref = segclip.Clipper().set_polygons(b, ovs)
    ref.build_tree().find_candidates()
    want, wc = _tree(ref), ref.counts()
    rings = O.Tree(b, ovs).clip(1, canonical=True).rings
    cl = segclip.Clipper()
    if again:  # the lists of other rings are there
        cl.set_polygons(S.star(300, 8), [S.star(200, 9, 0.1)])
        cl.build_tree().find_candidates()
    cl.set_polygons(b, ovs)
    for s in STAGES[:stages]:
        _call(cl, s)
    cl.clip(1)
    assert rings_equal(cl.rings(), rings) is None
    if again:
        got = _tree(cl)
    gc = cl.counts()
    for k in ("epc", "tree_size", "cover_entries", "leaf_end_entries", "tests", "candidates", "pairs", "stab_units",
              "near_pairs"):
        assert gc[k] == wc[k], k
    if not again:
        got = _tree(cl)
    assert all(np.array_equal(g, w) for g, w in zip(got, want))
    cl.clip(1)
    assert rings_equal(cl.rings(), rings) is None


def test_vertical_rings_after_some_stages(gpu):
    import segclip
    b, ovs = square(0.0, 0.0, 2.0, 2.0), [square(1.0, 0.5, 3.0, 1.5)]
    cl = segclip.Clipper().set_polygons(b, ovs)
    _call(cl, "elementary")
    cl.clip(1)  # the join refuses them, and the tree was not all there
    assert rings_equal(cl.rings(), O.Tree(b, ovs).clip(1, canonical=True).rings) is None


@pytest.mark.parametrize("stages", [0, 1, 2, 3])
def test_candidates_need_the_lists(gpu, stages):
    import segclip
    b, ovs = S.star1k()
    cl = segclip.Clipper().set_polygons(b, ovs)
    for s in STAGES[:stages]:
        _call(cl, s)
    with pytest.raises(segclip.SegclipError):
        cl.find_candidates()
    for s in STAGES[:3]:
        _call(cl, s)
    _call(cl, "cover_lists")
    cl.find_candidates()
    n = cl.counts()["pairs"]
    _call(cl, "elementary")  # the same points again: the lists stay good
    cl.find_candidates()
    assert cl.counts()["pairs"] == n == len(O.Tree(b, ovs).clip(1, canonical=True).pair_b)
