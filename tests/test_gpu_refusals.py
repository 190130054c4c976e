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


def _backward(cl, nb, nc):
    import segclip
    import torch
    g = torch.ones(1, dtype=torch.float64, device="cuda")
    gb, gc = (torch.zeros((n, 2), dtype=torch.float64, device="cuda") for n in (nb, nc))
    rc = segclip.lib().segclip_batch_area_backward_device(cl._h, *(C.c_void_p(t.data_ptr()) for t in (g, g, gb, gc)))
    return rc, gb.cpu().numpy(), gc.cpu().numpy()


# rings for the small-pair kernel and for the staged path
@pytest.mark.parametrize("nb,nc", [(40, 50), (300, 200)])
def test_gradients_of_a_batch_without_provenance(gpu, nb, nc):
    import segclip
    b, o = S.star(nb, 1, 0.0, 0.0, 0.5, 1.0), S.star(nc, 2, 0.1, 0.05, 0.5, 1.0)
    cl = segclip.Clipper().set_pairs([b], [o])
    cl.clip_batch()
    cl.set_provenance(True)
    assert _backward(cl, nb, nc)[0] == segclip._lib.ESTATE
    cl.clip_batch()
    rc, gb, gc = _backward(cl, nb, nc)
    assert rc == segclip._lib.OK and np.abs(gb).sum() > 0 and np.abs(gc).sum() > 0
    cl.release()
    assert _backward(cl, nb, nc)[0] == segclip._lib.ESTATE
    cl.clip_batch()
    again = _backward(cl, nb, nc)
    assert again[0] == segclip._lib.OK and np.allclose(again[1], gb) and np.allclose(again[2], gc)


def test_labelling_after_a_release(gpu):
    import segclip
    b, o = S.star(300, 1), S.star(200, 2, 0.1)
    cl = segclip.Clipper().set_polygons(b, [o])
    cl.clip(1)
    rings = cl.rings()
    area = cl.batch_area()
    cl.release()
    with pytest.raises(segclip.SegclipError) as e:
        cl.label_traverse()
    assert e.value.code == segclip._lib.ESTATE
    with pytest.raises(segclip.SegclipError):
        cl.intersections(1)
    assert np.array_equal(np.concatenate(cl.rings()), np.concatenate(rings))  # the last results stay
    assert np.array_equal(cl.batch_area(), area)
    cl.clip(1)
    assert np.array_equal(np.concatenate(cl.rings()), np.concatenate(rings))


def test_areas_and_labels_of_a_batch_of_other_rings(gpu):
    import segclip
    bases = [S.star(70 + k, k, 0.0, 0.0, 0.5, 1.0) for k in range(200)]
    ovs = [S.star(80 + k, 300 + k, 0.1, 0.05, 0.5, 1.0) for k in range(200)]
    cl = segclip.Clipper().set_pairs(bases, ovs).set_provenance(True)
    cl.clip_batch()
    rings = np.concatenate(cl.rings())
    cl.set_pairs(bases[:3], ovs[:3])
    for call in (cl.batch_area, cl.label_traverse, lambda: cl.intersections(1)):
        with pytest.raises(segclip.SegclipError) as e:
            call()
        assert e.value.code == segclip._lib.ESTATE
    assert _backward(cl, sum(map(len, bases[:3])), sum(map(len, ovs[:3])))[0] == segclip._lib.ESTATE
    assert np.array_equal(np.concatenate(cl.rings()), rings)
    assert len(cl.batch_status()) == 200
    cl.clip_batch()
    assert cl.batch_area().shape == (4, 3)
