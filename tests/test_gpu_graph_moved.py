"""GPU checks of calls after a graph replay that read other coordinates: clips,
pairs, counts and the tree then belong to the rings that the replay read, in a
context that had found pairs, or had built the tree, for earlier ones."""
import numpy as np
import pytest

import segclip.synth as S
from fixtures import rings_equal
from test_gpu_graph import _dev

pytestmark = pytest.mark.gpu

COUNTS = ("epc", "tree_size", "cover_entries", "leaf_end_entries", "tests", "candidates", "pairs")


def _rings(vertical):
    bases, ovs = S.small_pairs(60, 900)
    if vertical:  # the join refuses the batch
        bases[3][1, 0] = bases[3][0, 0]
    return bases, ovs, [o + np.array([0.05, 0.03]) for o in ovs]


def _replay(cl, bases, ovs):
    import torch
    bx, ox = _dev(bases, ovs)
    out = torch.empty((4, len(bases)), dtype=torch.float64, device="cuda")
    cl.pairs_area_graph(bx.data_ptr(), ox.data_ptr(), out.data_ptr())
    assert cl.get_tuning("small_fallback") == 0
    return bx, ox, out  # the graph's buffers


def _fresh(bases, ovs):
    import segclip
    ref = segclip.Clipper().set_pairs(bases, ovs).set_tuning("small_fused", 0)
    ref.clip_batch()
    return ref


@pytest.mark.parametrize("vertical", [False, True])
@pytest.mark.parametrize("before", ["clip", "tree", "stab"])
@pytest.mark.parametrize("first", ["clip", "pairs", "counts", "tree", "stages", "nothing found"])
def test_calls_after_a_replay_with_moved_rings(gpu, vertical, before, first):
    import segclip
    bases, ovs, moved = _rings(vertical)
    ref = _fresh(bases, moved)
    cl = segclip.Clipper().set_pairs(bases, ovs).set_tuning("small_fused", 0)
    if first != "nothing found":
        if before == "clip":
            cl.clip_batch()
        else:
            cl.build_tree()
            if before == "stab":
                cl.find_candidates()
    keep = _replay(cl, bases, moved)
    ks = range(1, len(bases) + 1)
    if first in ("clip", "nothing found"):
        cl.clip_batch()
    elif first == "pairs":
        for k in ks:
            assert all(np.array_equal(a, b) for a, b in zip(cl.pairs(k)[:2], ref.pairs(k)[:2])), k
    elif first == "counts":
        got, want = cl.counts(), ref.counts()
        assert all(got[c] == want[c] for c in COUNTS)
    elif first == "tree":
        assert np.array_equal(cl.cover_lists()[0], ref.cover_lists()[0])
        assert np.array_equal(cl.elementary(), ref.elementary())
    else:
        cl.find_candidates().intersections(7).label_traverse()
        ref2 = _fresh(bases, moved)
        ref2.intersections(7).label_traverse()
        assert rings_equal(cl.rings(), ref2.rings()) is None
    cl.clip_batch()
    got, want = cl.batch_rings(), ref.batch_rings()
    for k in ks:
        assert rings_equal(got[k - 1], want[k - 1]) is None, k
    assert all(np.array_equal(a, b) for k in ks for a, b in zip(cl.pairs(k)[:2], ref.pairs(k)[:2]))
    got, want = cl.counts(), ref.counts()
    assert all(got[c] == want[c] for c in COUNTS)
    del keep


def test_no_pairs_before_and_none_after(gpu):
    """A context that had found none refuses them after a replay as before it."""
    import segclip
    bases, ovs, moved = _rings(False)
    cl = segclip.Clipper().set_pairs(bases, ovs)
    cl.clip_batch()  # one launch, no pairs kept
    keep = _replay(cl, bases, moved)
    with pytest.raises(segclip.SegclipError):
        cl.pairs(1)
    with pytest.raises(segclip.SegclipError):
        cl.intersections(1)
    del keep
