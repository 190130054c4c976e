"""GPU check of rings with a common border of more pieces than the device-wide steps
of the sequential route list per job (256 chain starts): such a job runs in one
block, with the same rings; fewer pieces stay on the device-wide steps."""
import numpy as np
import pytest

import oracle_py as O
from fixtures import rings_equal

pytestmark = pytest.mark.gpu

STARTS = (3, 4)  # LEFT_ON, RIGHT_ON


def _layers(pieces):
    """A base below y = 0 and an overlay that follows the border for every third
    step and lies above it or below it between."""
    n = 3 * pieces
    x = np.arange(n + 1, dtype=np.float64)
    y = np.zeros(n + 1)
    y[2::3] = np.where(np.arange(len(y[2::3])) % 2 == 0, 0.25, -0.25)
    base = np.concatenate([np.stack([x[::-1], np.zeros(n + 1)], 1), [[-1.0, -6.0], [n + 1.0, -6.5]]])
    over = np.concatenate([np.stack([x[::-1], y[::-1]], 1), [[0.5, -5.0], [n - 0.5, -5.5]]])
    return base, over


@pytest.mark.parametrize("pieces", [200, 255, 256, 257, 258, 600])
def test_common_borders(gpu, pieces):
    import segclip
    base, over = _layers(pieces)
    print("[gpu-walk] common border of %d pieces" % pieces, flush=True)
    cl = segclip.Clipper().set_polygons(base, [over])
    got = []
    for par in (1, 0):
        cl.set_tuning("seq_parallel_walks", par).reset()
        cl.clip(1)
        lab = cl.augmented(0)[3]
        got.append((cl.rings(), cl.batch_status(), cl.batch_routes()))
    assert int(np.isin(lab, STARTS).sum()) == pieces
    assert rings_equal(got[0][0], got[1][0]) is None
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])
    assert rings_equal(got[0][0], O.Tree(base, [over]).clip(1, canonical=True).rings) is None
