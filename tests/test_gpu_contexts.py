"""Contexts that come and go: tables go up through pinned memory that outlives
the context and its stream, so a later context must neither wait on nor
overwrite anything of an earlier one."""
import threading

import numpy as np
import pytest

import segclip

pytestmark = pytest.mark.gpu


def _batch(count):
    """One base against 'count' small overlays in a context of its own: the output rings."""
    base = segclip.synth.star(500, count)
    ovs = [segclip.synth.star(8 + k % 5, k, 0.01 * (k % 60), 0.01 * (k % 40), 0.05, 0.1) for k in range(count)]
    cl = segclip.Clipper().set_polygons(base, ovs)
    cl.clip_batch(1, count)
    out = [np.concatenate(cl.rings()), np.asarray(cl.batch_status())]
    cl.close()
    return out


def _same(a, b):
    return len(a) == len(b) and all(x.shape == y.shape and (x == y).all() for x, y in zip(a, b))


# tables of a few words, beyond the first pinned block (256 KB) and within it again
@pytest.mark.parametrize("counts", [(2, 40, 3), (3, 30000, 2)])
def test_contexts_in_turn(counts):
    first = {n: _batch(n) for n in counts}
    for n in reversed(counts):
        assert _same(first[n], _batch(n))


def test_tables_beyond_the_pinned_memory():
    base, ov = segclip.synth.star(64, 1), segclip.synth.star(8, 2)
    n = 400000  # 5 MB of tables: copied, not staged
    cl = segclip.Clipper().set_polygons(base, [ov] * n)
    assert cl.counts()["num_edges"] == 64 + 8 * n
    cl.close()
    assert _same(_batch(2), _batch(2))


def test_contexts_on_threads():
    want = {n: _batch(n) for n in (2, 40, 3000)}
    bad = []

    def work(n):
        try:
            for _ in range(3):
                if not _same(want[n], _batch(n)):
                    bad.append(n)
        except Exception as e:  # reported by the caller
            bad.append(repr(e))

    for _ in range(2):  # the second set of threads takes over the first one's pinned memory
        ts = [threading.Thread(target=work, args=(n,)) for n in want]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    assert not bad


def test_context_after_a_failed_call():
    base, ov = segclip.synth.star(100, 5), segclip.synth.star(90, 6, 0.2, 0.1)
    want = None
    for turn in range(3):
        cl = segclip.Clipper()
        with pytest.raises(segclip.SegclipError):
            cl.set_polygons(base[:2], [ov])
        cl.set_polygons(base, [ov])
        with pytest.raises(segclip.SegclipError):
            cl.clip(2)
        cl.clip(1)
        got = [np.concatenate(cl.rings())]
        want = want or got
        assert _same(want, got)
        cl.close()
