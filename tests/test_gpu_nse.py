"""Table points of the cooling-table generator on the GPU (harm_nse.hpp):
three wavefronts per point against one thread per point, bit for bit, and both
against values of the one-integral-at-a-time chain that the reference's Fortran
fixes (every Newton solve run to its last trial), compiled for the host.

The solves stop at residuals of 1e-8 of a density and the outer one cycles at
the round-off of its central difference (a step of 1e-8: 1e-16 / 1e-8 on the
derivative), so an ulp of exp or pow moves the last iterate by up to about
1e-8 of the last step and no further: the bar is 1e-9."""
import ctypes

import numpy as np
import pytest

import harm_cool_amd as hc

pytestmark = pytest.mark.gpu

# (rho, T, HdFac) -> e, p, Qnu, tau, n_e-, n_e+: the corners of the table and
# points whose outer solve cycles (the first and fifth) and converges
POINTS = [
    ((1000000, 1000000000, 0.00062799999999999998),
     (8.3160700497303272e+22, 4.8218677295458038e+22, 1.0573353477816195e+19,
      4.8551114171653748e-14, 1.6181138716764039e-10, 1.4423809005285051e-15)),
    ((10000000000000, 1000000000, 0.00062799999999999998),
     (5.1975043160781823e+22, 2.7428239071110601e+22, 2521878501745527.5,
      1.1580054646065315e-17, 1.6181138716764039e-10, 1.4423809005285051e-15)),
    ((1000000, 1000000000000, 0.00062799999999999998),
     (3.4004670191661341e+34, 1.13431691546636e+34, 5.30565306110957e+39,
      169221.37618503574, 0.015209600295808328, 0.01520959999460351)),
    ((10000000000000, 1000000000000, 0.00062799999999999998),
     (3.5384567791090807e+34, 1.2175765181468157e+34, 9.6561212761375643e+38,
      700958.54729216942, 0.015292096533865535, 0.01512751505453073)),
    ((100000000, 5000000000, 0.5),
     (2.8730892913650364e+25, 1.5588338470962829e+25, 1.1535611589541265e+30,
      8.491867792339036e-06, 4.3918853280014488e-09, 4.7669376987733033e-10)),
    ((100000000000, 20000000000, 0.00062799999999999998),
     (9.2220845772096003e+28, 6.0414651220304522e+28, 3.8219453162912282e+35,
      0.015171945473244122, 1.5653661157427027e-07, 9.0989121304483209e-08)),
    ((1000000000, 200000000000, 0.00062799999999999998),
     (5.4203790684330075e+31, 1.8141563243733748e+31, 2.2859269439608373e+40,
      56.194492507585622, 0.00012180765957172855, 0.00012150664778975336)),
]


def _batch(fn, rho, T, hd):
    import torch

    ins = [torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device="cuda:0") for a in (rho, T, hd)]
    out = torch.full((6, len(rho)), -1.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    assert fn(*(ctypes.c_void_p(t.data_ptr()) for t in ins), ctypes.c_void_p(out.data_ptr()), len(rho), None) == 0
    return out.cpu().numpy()


@pytest.mark.parametrize("n", [1, 257])
def test_three_waves_equal_one_thread(n):
    rng = np.random.default_rng(n)
    rho, T, hd = 10 ** rng.uniform(6, 13, n), 10 ** rng.uniform(9, 12, n), 10 ** rng.uniform(-4, 0, n)
    a, b = (_batch(f, rho, T, hd) for f in (hc.lib().harm_eos_point_batch, hc.lib().harm_eos_point_batch_thread))
    assert np.isfinite(a).all()
    assert np.array_equal(a, b)


def test_points_match_serial_chain():
    ins = np.array([p[0] for p in POINTS]).T
    ref = np.array([p[1] for p in POINTS]).T
    got = _batch(hc.lib().harm_eos_point_batch, *ins)
    assert np.all(np.abs(got - ref) <= 1e-9 * np.abs(ref)), np.abs(got / ref - 1).max(axis=1)


def test_more_points_than_one_launch_holds():
    """2^32 threads and more: the points at the ends and at the launches' seams against
    a call of those alone (1e11 g/cm^3, 1e13 K: the shortest chains, 0.3 us a point)."""
    import torch

    n, span = 2 ** 32 // 192 + 1, 1 << 22
    at = torch.tensor([0, 1, 127, 128, span - 1, span, 3 * span - 1, 3 * span, n - 2, n - 1], device="cuda:0")
    few = [torch.full((len(at),), v, dtype=torch.float64, device="cuda:0") for v in (1e11, 1e13, 6.28e-4)]
    few[0] *= torch.linspace(0.5, 2.0, len(at), dtype=torch.float64, device="cuda:0")
    many = [torch.full((n,), v, dtype=torch.float64, device="cuda:0") for v in (1e11, 1e13, 6.28e-4)]
    many[0][at] = few[0]
    got = []
    for ins in (few, many):
        out = torch.full((6, len(ins[0])), -1.0, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        assert hc.lib().harm_eos_point_batch(*(ctypes.c_void_p(t.data_ptr()) for t in ins),
                                             ctypes.c_void_p(out.data_ptr()), len(ins[0]), None) == 0
        got.append(out)
    assert torch.equal(got[0], got[1][:, at])
    assert bool((got[1] > 0).all())
