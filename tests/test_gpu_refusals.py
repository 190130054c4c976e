"""GPU checks of calls on results that are not there: they are refused, with no
kernel run on memory that was never allocated, and the context goes on."""
import ctypes as C

import numpy as np
import pytest

import segclip.synth as S

pytestmark = pytest.mark.gpu


def _copy_rings(cl, pinned):
    import segclip
    import torch
    off = torch.empty(4, dtype=torch.int32, pin_memory=pinned)
    xy = torch.empty(8, dtype=torch.float64, pin_memory=pinned)
    rc = segclip.lib().segclip_copy_rings(cl._h, C.cast(off.data_ptr(), C.POINTER(C.c_int32)), 4,
                                          C.cast(xy.data_ptr(), C.POINTER(C.c_double)), 4, None)
    return rc


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("polygons", [False, True])
def test_rings_before_any_clip(gpu, pinned, polygons):
    import segclip
    cl = segclip.Clipper()
    b, o = S.star(50, 1), S.star(40, 2, 0.1)
    if polygons:
        cl.set_polygons(b, [o])
    assert _copy_rings(cl, pinned) == segclip._lib.ESTATE
    cl.set_polygons(b, [o])
    cl.clip(1)
    assert len(cl.rings()) > 0
