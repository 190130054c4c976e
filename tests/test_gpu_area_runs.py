"""GPU checks of the gradients summed per edge and per input vertex (rings that
belong to one job) against the ones added one by one (jobs that share their
base ring): edges with 1 to 5,000 crossings, so that the sums run over parts of
a wave, whole waves and many of them, on either side; ordinary rings; and rings
on a coarse sheared grid, whose output vertices come from shared vertices."""
import numpy as np
import pytest

import segclip.synth as S

pytestmark = pytest.mark.gpu

# A vertex sums at most 2 x 5,000 crossings' shares.  A share is at most the
# crossing's own gradient (the length of two output edges, below 8) over the sine
# of the angle between its edges (above 0.7 for the combs).  1e4 * 8 / 0.7 terms
# of size one, each rounded to 2^-53, stay below 2e-11.
TOL = 1e-10


def _comb(teeth, turn):
    t = np.arange(2 * teeth + 1)
    x = np.linspace(-1.0, 1.0, 2 * teeth + 1) + 0.2 / (2 * teeth + 1) * np.sin(2.1 * t)
    y = np.where(t % 2 == 1, 0.5, -0.5) + 0.05 * np.sin(1.3 * t)
    p = np.concatenate([np.stack([x, y], 1), [[1.3, -2.0], [-1.3, -2.1]]])
    return p[:, ::-1].copy() if turn else p


def _grid(ring, step):
    r = np.round(ring / step) * step
    return np.stack([r[:, 0] + r[:, 1] / 1024.0, r[:, 1]], 1)  # exact in double, no vertical edge


BAND = np.array([[-2.0, 0.013], [2.0, 0.017], [2.1, 3.0], [-2.1, 3.1]])
CASES = {
    "combs against a band": [(_comb(t, 0), BAND) for t in (1, 2, 3, 16, 31, 32, 33, 64, 250)],
    "a band against combs": [(BAND[:, ::-1].copy(), _comb(t, 1)) for t in (1, 31, 32, 33, 100, 1001)],
    "a long comb": [(_comb(2500, 0), BAND), (BAND, _comb(2500, 0))],
    "ordinary rings": [(S.star(300, 5), S.star(40, 6, 0.3, 0.1)), (S.harmonic(3000, 7), S.harmonic(900, 8, 0.1, 0.1)),
                       (S.star(9, 9), S.star(5, 10, 9.0, 9.0)), (S.star(9, 11, 0, 0, 0.1, 0.2), S.star(30, 12))],
    "rings on a grid": [(_grid(S.star(60 + 7 * k, 20 + k), 0.125), _grid(S.star(50 + 5 * k, 60 + k, 0.2, 0.1), 0.125))
                        for k in range(20)],
}


def _backward(cl, nb, nc, J):
    import torch
    ga = torch.linspace(0.5, 1.5, J, dtype=torch.float64, device="cuda")
    gi = torch.linspace(-1.0, 1.0, J, dtype=torch.float64, device="cuda")
    gb = torch.full((nb, 2), 7.0, dtype=torch.float64, device="cuda")
    gc = torch.full((nc, 2), 7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    cl.batch_area_backward_device(ga.data_ptr(), gi.data_ptr(), gb.data_ptr(), gc.data_ptr())
    return gb.cpu().numpy(), gc.cpu().numpy()


@pytest.mark.parametrize("name", sorted(CASES))
def test_summed_equals_added_one_by_one(gpu, name):
    import segclip
    for i, (b, o) in enumerate(CASES[name]):
        print("[gpu-area-runs] %s %d: %d x %d" % (name, i, len(b), len(o)), flush=True)
        far = S.star(12, 90, 50.0, 50.0)  # a second overlay, which makes the base ring a shared one
        shared = segclip.Clipper().set_polygons(b, [o, far]).set_provenance(True).clip_batch()
        if shared.batch_status()[0] & 1:
            continue  # undefined: some vertex has no slot
        pairs = segclip.Clipper().set_pairs([b, b], [o, far]).set_provenance(True).clip_batch()
        try:
            sb, sc = _backward(shared, len(b), len(o) + len(far), 2)
        except Exception as e:  # a vertex of the sequential route without provenance
            with pytest.raises(type(e)):
                _backward(pairs, 2 * len(b), len(o) + len(far), 2)
            continue
        pb, pc = _backward(pairs, 2 * len(b), len(o) + len(far), 2)
        pb = pb[:len(b)] + pb[len(b):]
        for s, p in ((sb, pb), (sc, pc)):
            assert np.max(np.abs(s - p)) <= TOL * max(1.0, np.max(np.abs(s)))
