"""GPU checks of the clean-up of nearly collinear vertices against the oracle
where its runs are long: sides cut into many collinear pieces (runs shorter
and longer than a window of 64 and a tile of 256 vertices, and longer than all
rounds reach, which one wave per ring then decides), rings that vanish
altogether, slowly bending rings where every few vertices one stays, and
many rings of both kinds next to one another."""
import math

import numpy as np
import pytest

import oracle_py as O
from fixtures import rings_equal

pytestmark = pytest.mark.gpu

BASE = np.array([[-3.0, -3.1], [3.2, -3.0], [3.05, 3.1], [-3.1, 3.0]])


def _cut_square(per_side, cx=0.0, cy=0.0, half=0.8, turn=0.3):
    c = np.array([[math.cos(turn + k * math.pi / 2), math.sin(turn + k * math.pi / 2)] for k in range(4)]) * half
    out = []
    for k in range(4):
        t = np.arange(per_side)[:, None] / per_side
        out.append(c[k] + t * (c[(k + 1) % 4] - c[k]))
    return np.concatenate(out) + [cx, cy]


def _circle(n, radius, cx=0.0, cy=0.0):
    t = 0.1 + 2 * math.pi * np.arange(n) / n
    return np.stack([cx + radius * np.cos(t), cy + radius * np.sin(t)], 1)


SHAPES = [_cut_square(p) for p in (1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1000, 20000)]
SHAPES += [_circle(n, r) for n, r in ((50, 1e-5), (700, 1e-3), (5000, 0.02), (20000, 0.5), (60000, 1.0))]


@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_long_runs_equal_the_oracle(gpu, i):
    import segclip
    ring = SHAPES[i]
    print("[gpu-cleanup] shape %d, %d vertices" % (i, len(ring)), flush=True)
    for shift in (0, 7):  # another root
        r = np.roll(ring, shift, axis=0)
        cl = segclip.Clipper().set_polygons(BASE, [r])
        cl.clip(1)
        err = rings_equal(cl.rings(), O.Tree(BASE, [r]).clip(1, canonical=True).rings)
        assert err is None, (shift, err)


def test_many_rings_in_one_batch(gpu):
    import segclip
    rng = np.random.default_rng(5)
    ovs = []
    for k in range(60):
        cx, cy = rng.uniform(-2, 2, 2)
        kind = k % 4
        if kind == 0:
            ovs.append(_cut_square(int(rng.integers(1, 400)), cx, cy, 0.3, rng.uniform(0.1, 1.4)))
        elif kind == 1:
            ovs.append(_circle(int(rng.integers(3, 900)), 10 ** rng.uniform(-5, -1), cx, cy))
        elif kind == 2:
            ovs.append(_cut_square(int(rng.integers(1, 12)), cx, cy, 2.5, rng.uniform(0.1, 1.4)))
        else:
            ovs.append(_circle(3, 0.2, cx, cy))
    print("[gpu-cleanup] %d overlays in one batch" % len(ovs), flush=True)
    cl = segclip.Clipper().set_polygons(BASE, ovs)
    cl.clip_batch()
    got = cl.batch_rings()
    tr = O.Tree(BASE, ovs)
    for k in range(len(ovs)):
        err = rings_equal(got[k], tr.clip(k + 1, canonical=True).rings)
        assert err is None, (k, err)
