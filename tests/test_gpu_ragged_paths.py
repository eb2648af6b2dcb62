"""Grids whose phi rows fill no wavefront, and 2D grids, on the step's other paths: the
learned and the gated Newton start and the capture of pairs against the plain step, the
tabulated EOS against the oracle."""
import ctypes

import numpy as np
import pytest

import harm_cool_amd as hc
from harm_cool_amd.params import torus_params
from oracle_lib import Oracle, lib as olib, orc_eos

pytestmark = pytest.mark.gpu

GRIDS = {"12x10x38": (12, 10, 38, {}), "2d": (24, 20, 1, {}), "9x11x6_ppm": (9, 11, 6, dict(lim=3)),
         "10x9x100_llf": (10, 9, 100, dict(lim=1, hllf=0.0, laxf=1.0))}


@pytest.mark.parametrize("grid", list(GRIDS))
def test_network_starts_match_the_plain_step(grid):
    """As on the wave-uniform grids: a gate that no first step reaches gives the plain
    step bit for bit; the network's starts (from pairs of the run's first steps; a low gate
    sends zones through the seed list) converge to the same roots, and the capture of pairs
    changes nothing."""
    import torch

    n1, n2, n3, kw = GRIDS[grid]
    P = torus_params(n1, n2, n3, **kw)
    cap = 4 * n1 * n2 * n3 + 5
    feat = torch.zeros((8, cap), dtype=torch.float64, device="cuda:0")
    targ = torch.zeros((2, cap), dtype=torch.float64, device="cuda:0")
    valid = torch.zeros(cap, dtype=torch.uint8, device="cuda:0")
    runs = {k: hc.Harm(P) for k in ("plain", "captured", "closed", "gated", "learned")}
    for s in runs.values():
        s.init()
    runs["captured"].set_capture(feat, targ, valid, 1)
    for k in ("plain", "captured"):
        runs[k].step_ch(2)
    assert np.array_equal(runs["plain"].prims(), runs["captured"].prims())
    assert runs["plain"].counters() == runs["captured"].counters()
    n = runs["captured"].capture_count()
    assert n == 4 * n1 * n2 * n3
    m = hc.Mlp(seed=3)
    fd, td, vd = feat[:, :n].contiguous(), targ[:, :n].contiguous(), valid[:n].contiguous()
    m.fit_norm(fd, td, vd)
    m.train(fd, td, vd, batch=2048, steps=200, lr0=3e-3, lr1=2e-4)
    runs["closed"].set_guess(2, m, gate=1e300)
    runs["gated"].set_guess(2, m, gate=1e-9)
    runs["learned"].set_guess(1, m)
    for k in ("closed", "gated", "learned"):
        runs[k].step_ch(2)
    for k, s in runs.items():
        s.step_ch(4)
    p0, c0 = runs["plain"].prims(), runs["plain"].counters()
    assert np.array_equal(runs["closed"].prims(), p0)
    assert runs["closed"].counters() == c0
    sl = (slice(None), slice(2, n1 + 2), slice(2, n2 + 2), slice(None))
    for k in ("gated", "learned"):
        p, c = runs[k].prims(), runs[k].counters()
        for v in range(8):
            x, y = p0[sl][v], p[sl][v]
            assert np.abs(x - y).max() <= 1e-10 * np.abs(x).max(), (k, v)
        assert c["newton_iters"] != c0["newton_iters"]  # other starts
        for name in ("c2p_calls", "fail_2d", "fixup_repairs", "fatal"):
            assert c[name] == c0[name], (k, name)
    for s in runs.values():
        s.close()
    m.close()


@pytest.mark.parametrize("n,kw,refd", [((12, 10, 38), {}, 0), ((12, 10, 38), dict(lim=1), 1),
                                       ((9, 11, 100), dict(lim=2, hllf=0.0, laxf=1.0), 0), ((10, 9, 6), dict(lim=3), 0),
                                       ((33, 18, 1), dict(lim=1), 0)])
def test_tabulated_steps_match_oracle(n, kw, refd):
    P = torus_params(*n, **kw)
    host = hc.eos_table_build(hc.eos_spec(rho_unit=1e8, nr=60, nt=50))
    tab = hc.DeviceEos(host, P.gam)
    g = hc.Harm(P)
    g.set_eos(tab, bool(refd))
    o = Oracle(P)
    olib().orc_set_threads(8)
    e = orc_eos(host, P.gam)
    olib().orc_set_eos(o.h, ctypes.byref(e), refd)
    g.init()
    o.init_torus()
    for s in range(4):
        g.step_ch(1)
        assert o.step() == 0
        assert g.time() == o.time(), s
        assert np.array_equal(g.prims(), o.prims()), s
        assert np.array_equal(g.pflag(), o.pflag()), s
        assert g.counters() == o.counters(), s
    g.close()
