"""The inversion in other units: density, energy and field scaled by powers of two scale
every operation exactly, so codes, iteration counts and the scaled primitives' bits must
not change -- over a range of units in which the divisions and roots of the kernels, which
leave out the scaling for operands at the ends of the exponent range, still hold."""
import os

import numpy as np
import pytest

import harm_cool_amd as hc

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "utoprim.npz")


@pytest.mark.parametrize("k", [-120, -40, 40])
def test_inversion_scales_exactly_with_the_units(k):
    import torch

    g = np.load(GOLD)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
    s, b = 2.0 ** k, 2.0 ** (k // 2)
    su = np.array([s] * 5 + [b] * 3)
    sp = np.array([s, s, 1., 1., 1., b, b, b])
    gcov, gcon, gdet, gam = dev(g["gcov"].T), dev(g["gcon"].T), dev(g["gdet"]), float(g["gam"])
    p1, p2 = dev(g["guess"].T), dev((g["guess"] * sp).T)
    r1 = hc.utoprim2d_batch(dev(g["U"].T), gcov, gcon, gdet, p1, gam)
    r2 = hc.utoprim2d_batch(dev((g["U"] * su).T), gcov, gcon, gdet, p2, gam)
    torch.cuda.synchronize()
    ok = (r1[0] == 0).cpu().numpy()
    assert ok.sum() > 100
    for a, c in zip(r1, r2):
        assert np.array_equal(a.cpu().numpy()[ok], c.cpu().numpy()[ok])
    assert np.array_equal((p1.cpu().numpy().T * sp)[ok], p2.cpu().numpy().T[ok])
