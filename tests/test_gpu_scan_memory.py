"""GPU check of device memory held by contexts that are gone: what they had per
stream of their own goes to later ones or back, however many were alive at once."""
import threading

import pytest

import segclip.synth as S
from fixtures import rings_equal

pytestmark = pytest.mark.gpu


def _held(count, base, ov, want=None):
    """Device bytes held after 'count' contexts that were alive at once, each with a side stream."""
    import segclip
    cls = [segclip.Clipper().set_polygons(base, [ov]).set_operation(True) for _ in range(count)]
    for cl in cls:
        cl.clip(1)
        assert want is None or rings_equal(cl.rings(), want) is None
    rings = cls[0].rings()
    for cl in cls:
        cl.close()
    return segclip.memory()[0], rings


def test_many_contexts_at_once(gpu):
    base, ov = S.harmonic(60000, 1), S.harmonic(70000, 2, 0.1, 0.1)
    first, want = _held(6, base, ov)
    # a context's scans of the four edge counts alone need a word for each of 35 + 35 + 30 + 30 tiles
    more, _ = _held(30, base, ov, want)
    assert more - first < 24 * 130 * 4 // 2
    assert _held(30, base, ov, want)[0] - more < 24 * 130 * 4 // 2


def test_contexts_closed_by_other_threads(gpu):
    import segclip
    base, ov = S.harmonic(6000, 1), S.harmonic(7000, 2, 0.1, 0.1)
    _, want = _held(1, base, ov)
    cls, bad = [], []

    def work():
        cl = segclip.Clipper().set_polygons(base, [ov]).set_operation(True)
        cl.clip(1)
        cls.append(cl)

    for _ in range(3):
        ts = [threading.Thread(target=work) for _ in range(4)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        while cls:
            cl = cls.pop()
            if rings_equal(cl.rings(), want) is not None:
                bad.append(1)
            cl.clip(1)  # here on this thread's scratch
            if rings_equal(cl.rings(), want) is not None:
                bad.append(2)
            cl.close()
    assert not bad
