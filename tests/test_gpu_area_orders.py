"""GPU checks that a job's areas do not depend on the batch it is in: rings of 3
to 256 vertices summed by a wave each (all rings that short) or by a block
(some ring longer), and jobs of 0 to 600 output rings added by a wave each (many
jobs) or by a block, give the same bits; output rings either side of the length
(4,096) that is summed in chunks agree with the shoelace in extended precision."""
import numpy as np
import pytest

import segclip.synth as S

pytestmark = pytest.mark.gpu

BAND = np.array([[-2.0, 0.013], [2.0, 0.017], [2.1, 3.0], [-2.1, 3.1]])


def _comb(teeth):
    t = np.arange(2 * teeth + 1)
    x = np.linspace(-1.0, 1.0, 2 * teeth + 1) + 0.2 / (2 * teeth + 1) * np.sin(2.1 * t)
    y = np.where(t % 2 == 1, 0.5, -0.5) + 0.05 * np.sin(1.3 * t)
    return np.concatenate([np.stack([x, y], 1), [[1.3, -2.0], [-1.3, -2.1]]])


def _clip(bases, ovs):
    import segclip
    cl = segclip.Clipper().set_pairs(bases, ovs)
    cl.set_tuning("small_fused", 0)
    return cl.clip_batch()


def _areas(bases, ovs):
    return np.asarray(_clip(bases, ovs).batch_area())


@pytest.mark.parametrize("teeth", [[1, 30], [64, 65, 126], [127, 255, 256, 257, 600]])
def test_areas_do_not_depend_on_the_batch(gpu, teeth):
    print("[gpu-area-orders] combs of %s teeth" % teeth, flush=True)
    bases = [_comb(t) for t in teeth] + [S.star(3, 5), S.star(64, 6), S.star(256, 7), S.star(9, 8)]
    ovs = [BAND] * len(teeth) + [S.star(65, 9, 0.1), S.star(3, 10, 0.2), S.star(255, 11, 0.1), S.star(5, 12, 9.0)]
    n = len(bases)
    alone = _areas(bases, ovs)
    many = _areas(bases + [S.star(5, 30 + i % 7) for i in range(2100)], ovs + [S.star(6, 40 + i % 5, 0.1) for i in range(2100)])
    longer = _areas(bases + [S.star(1000, 50)], ovs + [S.star(900, 51, 0.1)])
    assert np.array_equal(alone.view(np.uint64), many[:, :n].copy().view(np.uint64))
    assert np.array_equal(alone.view(np.uint64), longer[:, :n].copy().view(np.uint64))


@pytest.mark.parametrize("n", [300, 4095, 4096, 4097, 9000])
def test_long_output_rings(gpu, n):
    print("[gpu-area-orders] output ring of %d vertices" % n, flush=True)
    ring = S.star(n, 60 + n, 0.0, 0.0, 0.9, 1.0)
    box = np.array([[-3.0, -3.1], [3.2, -3.0], [3.0, 3.1], [-3.1, 3.0]])
    cl = _clip([box, box], [ring, S.star(7, 3)])
    got, (out,) = np.asarray(cl.batch_area()), cl.batch_rings()[0]
    assert n - 30 <= len(out) <= n  # the clean-up may drop nearly collinear vertices
    x, y = out[:, 0].astype(np.longdouble), out[:, 1].astype(np.longdouble)
    want = abs(np.sum(x * np.roll(y, -1) - np.roll(x, -1) * y)) / 2
    # n terms below 2.1 in size, each product and partial sum rounded to 2^-53
    assert abs(float(got[0, 0] - want)) <= 2.1 * n * 4 * 2.0 ** -53 * max(1.0, np.log2(n))


@pytest.mark.parametrize("combs", [13, 14])  # 600 output rings each: 7,800 and 8,400 with 8,192 waves to take them
def test_output_rings_one_or_four_a_wave(gpu, combs):
    print("[gpu-area-orders] %d combs of 600 teeth" % combs, flush=True)
    bases, ovs = [S.star(300, 21), S.star(17, 22), _comb(40)], [S.star(200, 23, 0.1), S.star(9, 24, 0.1), BAND]
    alone = _areas(bases, ovs)
    many = _areas(bases + [_comb(600)] * combs, ovs + [BAND] * combs)
    assert np.array_equal(alone.view(np.uint64), many[:, :3].copy().view(np.uint64))
    assert len(set(many[0, 3:].tolist())) == 1
