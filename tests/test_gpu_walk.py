"""GPU checks of the sequential labelling route run over the whole device
against its single walk ("seq_parallel_walks" = 0, one lane per job): rings,
status and route bit for bit, for unions, rings on a coarse grid (touching
and overlapping edges, split bouncing pairs, chains, walks that never close)
and sizes either side of the node count where the device-wide steps start."""
import numpy as np
import pytest

import oracle_py as O
import segclip.synth as S
from fixtures import rings_equal

pytestmark = pytest.mark.gpu


def _grid(ring, step):
    return np.round(ring / step) * step if step else ring


CASES = [
    # (union, base, overlay, grid step)
    (True, S.harmonic(8009, 11), S.harmonic(21001, 12, 0.15, -0.1, 1.0, 0.3), 0.0),
    (True, S.star(700, 13), S.star(700, 14, 0.2, 0.1), 0.0),    # about 2,000 nodes
    (True, S.star(1500, 15), S.star(1700, 16, 0.2, 0.1), 0.0),  # well above
    (False, S.harmonic(20000, 17), S.harmonic(50000, 18, 0.15, -0.1, 1.0, 0.3), 0.0005),
    (False, S.harmonic(20000, 19), S.harmonic(50000, 20, 0.15, -0.1, 1.0, 0.3), 0.0003),
    (False, S.harmonic(12000, 21), S.harmonic(30000, 22, 0.1, 0.1, 1.0, 0.2), 0.0002),
    (True, S.harmonic(12000, 23), S.harmonic(30000, 24, 0.1, 0.1, 1.0, 0.2), 0.0003),
    (False, S.harmonic(40000, 25), S.harmonic(90000, 26, 0.1, -0.1, 1.0, 0.2), 0.0001),
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_device_wide_steps_equal_the_single_walk(gpu, i):
    import segclip
    uni, b, c, step = CASES[i]
    print("[gpu-walk] case %d: union %d, %d x %d, grid %g" % (i, uni, len(b), len(c), step), flush=True)
    cl = segclip.Clipper().set_polygons(_grid(b, step), [_grid(c, step)])
    cl.set_operation(uni)
    got = []
    for par in (1, 0):
        cl.set_tuning("seq_parallel_walks", par)
        for _ in range(2):  # the second on buffers that hold the first's leftovers
            cl.reset()
            cl.clip(1)
        got.append((cl.rings(), cl.batch_status(), cl.batch_routes()[0]))
    err = rings_equal(got[0][0], got[1][0])
    assert err is None, err
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])
    if uni and not step:
        assert rings_equal(got[0][0], O.Tree(b, [c]).clip(1, canonical=True, union=True).rings) is None


def test_batch_with_unions_of_every_size(gpu):
    import segclip
    base = S.harmonic(30000, 31)
    ovs = [S.star(n, 60 + n, 0.3 - 0.05 * k, 0.1 * k, 0.2, 0.6) for k, n in enumerate((12, 300, 2500, 9000, 15001))]
    ovs.append(S.star(50, 5, 9.0, 9.0, 0.5, 1.0))  # disjoint: a union of two rings
    print("[gpu-walk] one base, %d unions" % len(ovs), flush=True)
    cl = segclip.Clipper().set_polygons(base, ovs).set_operation(True)
    cl.clip_batch()
    got, st = cl.batch_rings(), cl.batch_status()
    cl.set_tuning("seq_parallel_walks", 0)
    cl.reset()
    cl.clip_batch()
    want = cl.batch_rings()
    assert np.array_equal(st, cl.batch_status())
    for g, w in zip(got, want):
        assert rings_equal(g, w) is None
