"""GPU checks of one-to-many batches in which a base edge has more intersections
than the ordering inside groups takes (4,096): the labelling's first kernels run
before that is known, on positions that must then hold no slot, whatever an
earlier batch left in their memory.  The earlier batches have base rings of
thousands of edges, the batch under test one of four."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S
from fixtures import rings_equal
from test_gpu_runs import _comb

pytestmark = pytest.mark.gpu

BASE = np.array([[-2.0, -1.01], [2.0, -1.0], [2.02, 1.0], [-2.03, 1.02]])


def _earlier(cl):
    """A batch with more positions than the one under test, on edges that its base ring does not have."""
    cl.set_polygons(S.star(6000, 3), [S.star(6000, 4, 0.05, 0.02), S.star(5000, 5, -0.03, 0.04)])
    cl.clip_batch()
    assert sum(len(cl.pairs(k)[0]) for k in (1, 2)) > 20000


def _check(cl, ovs, want):
    cl.set_polygons(BASE, ovs)
    cl.clip_batch()
    got = cl.batch_rings()
    for k, w in enumerate(want):
        err = rings_equal(got[k], w)
        assert err is None, "overlay %d: %s" % (k + 1, err)


@pytest.mark.parametrize("teeth", [(2049, 30), (30, 2500), (2100, 2200)])
def test_large_group_after_a_larger_base(gpu, teeth):
    import segclip
    print("[gpu-slots] combs of %s teeth" % (teeth,), flush=True)
    ovs = [_comb(t, -1.0 if i == 0 else 1.0, i) for i, t in enumerate(teeth)] + [S.star(20, 9, 8.0, 8.0)]
    tree = O.Tree(BASE, ovs)
    want = [tree.clip(k, canonical=True).rings for k in range(1, len(ovs) + 1)]
    cl = segclip.Clipper()
    _earlier(cl)
    _check(cl, ovs, want)  # the context's own buffers
    cl.close()
    with segclip.torch_allocator():  # blocks that another context gave back
        cl = segclip.Clipper()
        _earlier(cl)
        cl.close()
        cl = segclip.Clipper()
        _check(cl, ovs, want)
        cl.close()
