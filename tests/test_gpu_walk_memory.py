"""GPU checks of the memory of the sequential route over the whole device: only jobs
that are large enough for it have scratch there, and where there is no memory for
that the jobs run in one block each, with the same rings."""
import ctypes as C

import numpy as np
import pytest

import segclip.synth as S
from fixtures import rings_equal

pytestmark = pytest.mark.gpu

PER_JOB = 2048 * 96 + 4096 * 16 + 3 * 256 * 8  # bytes of a walking job's lists


def _clip(bases, ovs, par=1):
    import segclip
    cl = segclip.Clipper().set_pairs(bases, ovs).set_operation(True).set_tuning("seq_parallel_walks", par)
    cl.clip_batch()
    return cl


def test_small_jobs_beside_a_large_one(gpu):
    import segclip
    n = 4096
    bases = [S.star(8 + k % 5, k) for k in range(n)]
    ovs = [S.star(9, 7 * k, 0.1, 0.1) for k in range(n)]
    bases[5], ovs[5] = S.star(1500, 1), S.star(1400, 2, 0.1, 0.1)
    cl = _clip(bases, ovs, 0)
    want, status = cl.batch_rings(), cl.batch_status()
    cl.release().close()
    start = segclip.memory(True)[0]
    cl = _clip(bases, ovs)
    peak = segclip.memory()[1]
    got = cl.batch_rings()
    print("[gpu-walk] %d jobs, one large: %d MiB" % (n, (peak - start) >> 20), flush=True)
    assert all(rings_equal(g, w) is None for g, w in zip(got, want))
    assert np.array_equal(cl.batch_status(), status)
    assert peak - start < n * PER_JOB // 2  # all else takes a tenth of that
    cl.release().close()


def test_no_memory_for_the_walks(gpu):
    import segclip
    import torch
    n, limit = 64, 64 * 2048 * 96  # the terms, and no other buffer of this batch
    bases = [S.star(600 + k, k) for k in range(n)]
    ovs = [S.star(500 + k, 100 + k, 0.1, 0.1) for k in range(n)]
    cl = _clip(bases, ovs, 0)
    want, status = cl.batch_rings(), cl.batch_status()
    cl.release().close()
    refused = []

    def alloc(nbytes, _user):
        if nbytes >= limit:
            refused.append(nbytes)
            return None
        return torch.cuda.caching_allocator_alloc(int(nbytes), 0)

    def free(ptr, _user):
        torch.cuda.caching_allocator_delete(ptr)

    hooks = segclip._ALLOC_FN(alloc), segclip._FREE_FN(free)
    torch.cuda.init()
    L = segclip.lib()
    assert L.segclip_set_allocator(C.cast(hooks[0], C.c_void_p), C.cast(hooks[1], C.c_void_p), None) == 0
    try:
        cl = _clip(bases, ovs)
        got, st = cl.batch_rings(), cl.batch_status()
        cl.release().close()
    finally:
        L.segclip_set_allocator(None, None, None)
        test_no_memory_for_the_walks.hooks = hooks  # scratch of the thread may come from them
    assert len(refused) == 1
    assert all(rings_equal(g, w) is None for g, w in zip(got, want))
    assert np.array_equal(st, status)
