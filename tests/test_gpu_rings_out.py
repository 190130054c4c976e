"""GPU checks of segclip_copy_rings: the same offsets and coordinates in
pinned memory, at an offset inside it, in ordinary memory and at addresses
that are only 8-byte aligned, for results of no ring, a few KB (written by a
kernel), either side of the staged and direct limits, and more than one
2-million-vertex piece."""
import ctypes as C

import numpy as np
import pytest

import segclip.synth as S

pytestmark = pytest.mark.gpu


def _copy(cl, off, xy, n_off, n_xy):
    from segclip import lib
    need = (C.c_int64 * 2)()
    rc = lib().segclip_copy_rings(cl._h, C.cast(off, C.POINTER(C.c_int32)), n_off, C.cast(xy, C.POINTER(C.c_double)),
                                  n_xy, need)
    assert rc == 0


# overlay sizes inside one large base per pair: the output is the overlays
@pytest.mark.parametrize("sizes", [None, [5], [3000], [16000], [20000, 5], [270000], [1200000, 1300001]])
def test_copy_rings_to_any_host_memory(gpu, sizes):
    import torch
    import segclip
    print("[gpu-rings-out]", sizes, flush=True)
    base = np.array([[-3.0, -3.1], [3.2, -3.0], [3.0, 3.1], [-3.1, 3.0]])
    if sizes is None:  # disjoint: no ring
        cl = segclip.Clipper().set_polygons(base, [S.star(10, 1, 9.0, 9.0)])
        cl.clip(1)
        want_off, want = np.zeros(1, np.int32), np.zeros((0, 2))
    else:
        ovs = [S.star(n, 40 + i) for i, n in enumerate(sizes)]
        cl = segclip.Clipper().set_pairs([base] * len(ovs), ovs)
        cl.set_tuning("small_fused", 0)
        cl.clip_batch()
        want_off, want = None, None
    from segclip import lib
    need = (C.c_int64 * 2)()
    lib().segclip_copy_rings(cl._h, None, 0, None, 0, need)
    no, nv = need[0], need[1]
    for kind in ("plain", "pinned", "pinned inside", "plain odd", "pinned odd"):
        off = torch.full((no + 8,), -7, dtype=torch.int32, pin_memory=kind.startswith("pinned"))
        xy = torch.full((2 * nv + 9,), -7.0, dtype=torch.float64, pin_memory=kind.startswith("pinned"))
        s_off, s_xy = (0, 0) if kind in ("plain", "pinned") else ((3, 4) if "inside" in kind else (1, 1))
        _copy(cl, off.data_ptr() + 4 * s_off, xy.data_ptr() + 8 * s_xy, no, nv)
        o, v = off[s_off:s_off + no].numpy().copy(), xy[s_xy:s_xy + 2 * nv].numpy().reshape(-1, 2).copy()
        if want is None:
            want_off, want = o, v
            assert nv > 0 and o[0] == 0 and o[-1] == nv
            assert sorted(map(tuple, v[:50])) and np.isin(v[:, 0], np.concatenate([r[:, 0] for r in ovs])).all()
        assert np.array_equal(o, want_off) and np.array_equal(v, want), kind
        # nothing outside the destination is written
        assert (off[s_off + no:] == -7).all() and (xy[s_xy + 2 * nv:] == -7.0).all()
        assert (off[:s_off] == -7).all() and (xy[:s_xy] == -7.0).all()
    assert len(cl.rings()) == no - 1
