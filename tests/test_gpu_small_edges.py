"""GPU checks of the one-wave-per-pair kernel at its edges against the staged
path and the oracle: two combs across each other with intersection counts
either side of a wave (64) and of the capacity (128, beyond it the staged path
takes over), rings of 3 and of 64 vertices, rings inside one another, and
rings on a coarse sheared grid (no vertical edge), a batch each, whose touching
vertices and overlapping edges the kernel either clips or hands on."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S
from fixtures import rings_equal

pytestmark = pytest.mark.gpu


def _comb(teeth, turn):
    """Slanted teeth from -1.5 to 1.5 between -1 and 1, closed on one side; turned by a quarter."""
    t = np.arange(2 * teeth + 1)
    along = np.linspace(-1.0, 1.0, 2 * teeth + 1) + 0.003 * np.sin(2.3 * t)
    across = np.where(t % 2 == 1, 1.5, -1.5) + 0.02 * np.sin(1.1 * t + turn)
    p = np.concatenate([np.stack([along, across], 1), [[1.3, -2.5], [-1.35, -2.6]]])
    return np.stack([-p[:, 1], p[:, 0]], 1) if turn else p


def _both(base, ov):
    import segclip
    out = []
    for fused in (1, 0):
        cl = segclip.Clipper().set_pairs([base], [ov])
        cl.set_tuning("small_fused", fused)
        cl.clip_batch()
        out.append((cl.batch_rings()[0], cl.batch_status(), cl.batch_area(), cl.get_tuning("small_fallback")))
    assert rings_equal(out[0][0], out[1][0]) is None
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2].view(np.uint64), out[1][2].view(np.uint64))
    r = O.Tree(base, [ov]).clip(1, canonical=True)
    if not r.status & 1:
        assert rings_equal(out[0][0], r.rings) is None
    return out[0][3], len(out[0][0])


@pytest.mark.parametrize("a,b", [(1, 1), (3, 5), (4, 4), (16, 1), (1, 17), (17, 1), (30, 1), (1, 30), (4, 8), (8, 4), (3, 11),
                                 (11, 3), (30, 30)])
def test_combs_across_each_other(gpu, a, b):
    print("[gpu-small-edges] combs of %d and %d teeth" % (a, b), flush=True)
    fell, rings = _both(_comb(a, 0), _comb(b, 1))
    assert rings > 0
    assert (fell != 0) == (4 * a * b > 128)


@pytest.mark.parametrize("n,m", [(3, 3), (3, 64), (64, 3), (64, 64), (63, 62), (32, 33)])
def test_ring_sizes(gpu, n, m):
    print("[gpu-small-edges] rings of %d and %d vertices" % (n, m), flush=True)
    for k, (dx, lo) in enumerate(((0.2, 0.5), (0.0, 0.02), (5.0, 0.5))):
        b, o = S.star(n, 300 + n, 0.0, 0.0, 0.5, 1.0), S.star(m, 400 + m, dx, 0.1 * dx, lo, 2 * lo)
        fell, rings = _both(b, o)
        if n > 5 and m > 5 and k:
            assert fell == 0 and rings == (1 if k == 1 else 0)


@pytest.mark.parametrize("step", [0.5, 0.25, 0.125, 0.0625])
def test_rings_on_a_grid(gpu, step):
    kept = 0
    for seed in range(40):
        b, o = (np.round(r / step) * step for r in (S.star(5 + seed % 23, 500 + seed, 0.0, 0.0, 0.5, 1.0),
                                                    S.star(4 + seed % 17, 600 + seed, 0.2, 0.1, 0.5, 1.0)))
        b, o = (np.stack([r[:, 0] + r[:, 1] / 1024.0, r[:, 1]], 1) for r in (b, o))  # exact in double
        print("[gpu-small-edges] grid %g seed %d" % (step, seed), flush=True)
        fell, _ = _both(b, o)
        kept += fell == 0
    if step < 0.2:
        assert kept > 0
