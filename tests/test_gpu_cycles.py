"""GPU checks of the crossing cycles' minima and distances against the oracle
either side of the count (4,096 crossings of the base side) up to which one
block finds them: a comb cut by a band below its tips (all crossings on one
cycle) and by one above its gaps (two crossings per cycle)."""
import numpy as np
import pytest

import oracle_py as O
from fixtures import rings_equal

pytestmark = pytest.mark.gpu


def _comb(teeth):
    """Tips at y = 1 and gaps at y = -1, closed far below."""
    t = np.arange(2 * teeth + 1)
    x = np.linspace(-1.0, 1.0, 2 * teeth + 1) + 0.1 / (2 * teeth) * np.sin(t)
    y = np.where(t % 2 == 1, 1.0, -1.0) + 0.05 * np.sin(1.7 * t)
    return np.concatenate([np.stack([x, y], 1), [[1.2, -4.0], [-1.25, -4.1]]])


@pytest.mark.parametrize("teeth", [1, 2, 31, 512, 1023, 1024, 1025, 2047, 2048, 2049, 3000])
@pytest.mark.parametrize("above", [False, True])
def test_comb_cut_by_a_band(gpu, teeth, above):
    import segclip
    print("[gpu-cycles] %d teeth, %s" % (teeth, "above" if above else "below"), flush=True)
    band = np.array([[-2.0, 0.013], [2.0, 0.017], [2.1, 3.0], [-2.1, 3.1]]) if above else \
        np.array([[-2.0, -2.0], [2.0, -2.1], [2.1, 0.017], [-2.1, 0.013]])
    base = _comb(teeth)
    cl = segclip.Clipper().set_polygons(base, [band])
    cl.clip(1)
    got = cl.rings()
    assert len(got) == (teeth if above else 1)
    err = rings_equal(got, O.Tree(base, [band]).clip(1, canonical=True).rings)
    assert err is None, err
