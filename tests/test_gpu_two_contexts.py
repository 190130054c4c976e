"""GPU checks of two live contexts, each with a stream of its own, used in turn by
one host thread: the scratch of a call belongs to the thread, so a call's work is
done with it on return, and no call changes what another context holds."""
import numpy as np
import pytest

import segclip.synth as S
from fixtures import degenerate_cases, rings_equal
from test_gpu_graph import _dev, _eager

pytestmark = pytest.mark.gpu


def _pairs(n, seed, fused=1):
    import segclip
    bases, ovs = S.small_pairs(n, seed)
    return segclip.Clipper().set_pairs(bases, ovs).set_tuning("small_fused", fused)


def _far(n):
    """Overlays that meet no base: nothing to put out."""
    import segclip
    return segclip.Clipper().set_polygons(S.star(50, n), [S.star(9, k, 20.0 + k, 9.0) for k in range(n)])


# small batches in one launch, batches on the staged path, batches without output
@pytest.mark.parametrize("make", [
    lambda i: _pairs((3000, 2500, 40)[i], 70 + i), lambda i: _pairs((400, 700, 40)[i], 80 + i, i % 2),
    lambda i: _far(5) if i == 1 else _pairs(300, 90 + i, i % 2)])
def test_batches_in_turn(gpu, make):
    want = []
    for i in range(3):
        cl = make(i)
        cl.clip_batch()
        want.append((cl.batch_rings(), cl.batch_area()))
        cl.close()
    cls = [make(i) for i in range(3)]
    for turn in range(4):
        order = [(turn + q) % 3 for q in range(3)]
        for i in order:
            cls[i].clip_batch()
        for i in order:  # nothing was read before the others had run
            got = cls[i].batch_rings()
            assert len(got) == len(want[i][0])
            assert all(rings_equal(g, w) is None for g, w in zip(got, want[i][0])), (turn, i)
            assert np.array_equal(cls[i].batch_area(), want[i][1])
    for cl in cls:
        cl.close()


def test_graphs_with_uncovered_pairs_in_turn(gpu):
    import segclip
    import torch
    cls = []
    for seed in (5200, 5300):
        bases, ovs = S.small_pairs(64, seed)
        for _, b, o, _ in degenerate_cases():
            if len(b) <= 64 and len(o[0]) <= 64:
                bases.append(b)
                ovs.append(o[0])
        bx, ox = _dev(bases, ovs)
        cl = segclip.Clipper().set_pairs_device(bx.data_ptr(), [len(b) for b in bases], ox.data_ptr(),
                                                [len(o) for o in ovs])
        cls.append((cl, bx, ox, torch.empty((4, len(bases)), dtype=torch.float64, device="cuda"), _eager(bases, ovs)))
    for _ in range(3):
        for cl, bx, ox, out, want in cls:
            cl.pairs_area_graph(bx.data_ptr(), ox.data_ptr(), out.data_ptr())
        for cl, bx, ox, out, want in cls:
            assert np.array_equal(out.cpu().numpy().view(np.uint64), want.view(np.uint64))
