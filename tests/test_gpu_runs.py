"""GPU checks of the order of a shared base ring's intersections along its
edges, which one-to-many batches take from the runs of pairs of one edge: edges
with numbers of intersections either side of a thread's (8), a wave's (64, 512)
and a block's share (4,096; beyond it one sort orders the pairs), several such
edges per job, mixed with jobs of none."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S
from fixtures import rings_equal

pytestmark = pytest.mark.gpu


def _comb(teeth, y0, phase):
    """A comb of the given number of teeth across y = y0, between x = -1 and 1."""
    n = 2 * teeth + 1
    t = np.arange(n)
    x = np.linspace(-1.0, 1.0, n) + 0.2 / n * np.sin(2.1 * t + phase)
    y = y0 + np.where(t % 2 == 1, 0.3, -0.3) + 0.05 * np.sin(1.3 * t + phase)
    return np.concatenate([np.stack([x, y], 1), [[1.3, y0 - 0.8], [-1.3, y0 - 0.83]]])[::-1 if phase > 2 else 1]


@pytest.mark.parametrize("sizes", [(4, 5, 3), (8, 9, 31), (32, 33, 255), (256, 257, 300), (2047, 2048, 5), (2049, 7, 2500)])
def test_intersections_along_long_edges(gpu, sizes):
    import segclip
    base = np.array([[-2.0, -1.01], [2.0, -1.0], [2.02, 1.0], [-2.03, 1.02]])  # two edges take all crossings
    ovs = []
    for i, t in enumerate(sizes):
        ovs += [_comb(t, -1.0, i), S.star(20, 70 + i, 8.0, 8.0), _comb(t + 1, 1.0, i + 2.5)]
    ovs.append(S.harmonic(500, 5, 0.1, 0.1, 1.0, 0.3))
    print("[gpu-runs] combs of %s teeth" % (sizes,), flush=True)
    cl = segclip.Clipper().set_polygons(base, ovs)
    cl.clip_batch()
    got = cl.batch_rings()
    tree = O.Tree(base, ovs)
    for k in range(1, len(ovs) + 1):
        err = rings_equal(got[k - 1], tree.clip(k, canonical=True).rings)
        assert err is None, "overlay %d: %s" % (k, err)
