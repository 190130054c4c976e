"""GPU checks of the candidate pairs' order either side of the counts where
their sort changes: a wave's run (512), a block of places (1,024) and the end
of the two-launch sort (16,384), for one overlay, several and pairs."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S

pytestmark = pytest.mark.gpu


def _comb(edges):
    """A zigzag of the given number of edges across y = 0, closed far below."""
    t = np.arange(edges + 1)
    x = np.linspace(-1.0, 1.0, edges + 1) + 0.1 / edges * np.sin(t)
    y = np.where(t % 2 == 1, 1.0, -1.0) + 0.05 * np.sin(1.7 * t)
    end = [[1.2, y[-1] - 0.01], [1.21, -4.0], [-1.25, -4.1], [-1.2, -1.4]]
    return np.concatenate([np.stack([x, y], 1), end])


BAND = np.array([[-2.0, 0.013], [2.0, 0.017], [2.1, 3.0], [-2.1, 3.1]])


@pytest.mark.parametrize("n", [2, 510, 512, 514, 1022, 1024, 1026, 4096, 8192, 16382, 16384, 16386, 20000])
def test_pair_order(gpu, n):
    import segclip
    base = _comb(n)  # an even number of edges: the last one ends below the band
    print("[gpu-sort-sizes] %d pairs" % n, flush=True)
    cl = segclip.Clipper().set_polygons(base, [BAND])
    cl.clip(1)
    b, c, t = cl.pairs(1)
    r = O.Tree(base, [BAND]).clip(1, canonical=True)
    assert len(b) == n and np.array_equal(b, r.pair_b) and np.array_equal(c, r.pair_c) and np.array_equal(t, r.pair_type)


@pytest.mark.parametrize("paired", [False, True])
@pytest.mark.parametrize("half", [256, 4096, 8192, 8194])
def test_pair_order_of_two_jobs(gpu, half, paired):
    import segclip
    base, ovs = _comb(half), [BAND, BAND + [0.0, 0.1]]
    print("[gpu-sort-sizes] two times %d pairs, %s" % (half, "paired" if paired else "shared"), flush=True)
    cl = segclip.Clipper()
    if paired:
        cl.set_pairs([base, base], ovs).set_tuning("small_fused", 0)
    else:
        cl.set_polygons(base, ovs)
    cl.clip_batch()
    rings = cl.batch_rings()
    for k, o in enumerate(ovs):
        want = O.Tree(base, [o]).clip(1, canonical=True).rings
        assert len(rings[k]) == len(want)
        for g, w in zip(rings[k], want):
            assert np.array_equal(g, w)
