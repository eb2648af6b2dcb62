"""What a cache holds on the device: the values alone until it is looked up (a run with one
cache per radius keeps hundreds that never are), then the table of its splines; the table's
first use from several threads and streams at once."""
import threading

import numpy as np
import pytest

import ceos_cases as cc
import harm_cool_amd as hc
from harm_cool_amd.params import torus_params
from test_gpu_cache import random_cache

pytestmark = pytest.mark.gpu


def _used():
    import torch

    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_step_caches_hold_no_lookup_table():
    """The device's memory for one 128x128x5 cache per radius and the step that runs on
    them: the values (0.7 MB each) and the context's splines of e and p (3.1 MB), each
    allocation rounded to at most 2 MB more; a lookup table would be 7.9 MB."""
    import torch

    rho, T, v = cc.gas_rad(128, 128)
    d = hc.cache_desc(128, rho[0], rho[-1], 128, T[0], T[-1], d=5, whole=1)
    P = torus_params(28, 8, 1)
    g = hc.Harm(P)
    g.init()
    torch.zeros(1, device="cuda:0")
    m0 = _used()
    caches = [hc.Cache.create(d, rho, T, np.array([1.]), v, np.ones((1, 128, 128), np.uint8))
              for _ in range(P.n1 + 4)]
    g.set_eos_cache(caches)
    g.step_ch(1)
    per = (_used() - m0) / len(caches)
    assert per < 8.2e6, per
    x = torch.tensor([1e6], dtype=torch.float64, device="cuda:0")
    zi = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    m1 = _used()
    for c in caches:
        c.lookup(x, x, None, zi)
    assert (_used() - m1) / len(caches) > 7.5e6  # and the tables once they are looked up
    for c in caches:
        c.close()
    g.close()


def test_first_lookups_from_several_threads():
    import torch

    rng = np.random.default_rng(5)
    for _ in range(4):
        arrays = random_cache(rng, X=40, Y=50, Z=2, D=3, types=(hc.AXIS_LOG, hc.AXIS_LOG, hc.AXIS_LINEAR))
        desc, vx, vy = arrays[:3]
        q = 3000
        x = torch.from_numpy(np.exp(rng.uniform(np.log(vx[0]), np.log(vx[-1]), q))).to("cuda:0")
        y = torch.from_numpy(np.exp(rng.uniform(np.log(vy[0]), np.log(vy[-1]), q))).to("cuda:0")
        zi = torch.from_numpy(rng.integers(0, 2, q).astype(np.int32)).to("cuda:0")
        want = hc.Cache.create(*arrays)
        ref = want.lookup(x, y, None, zi, dery=True)
        shared = hc.Cache.create(*arrays)
        got, start = [None] * 6, threading.Barrier(6)

        def work(k):
            L = hc.lib()
            s = torch.cuda.Stream()
            o = [torch.full((3, q), float("nan"), dtype=torch.float64, device="cuda:0") for _ in range(2)]
            st = torch.full((q,), -1, dtype=torch.int32, device="cuda:0")
            torch.cuda.synchronize()
            start.wait()
            rc = L.harm_cache_lookup(shared.h, hc.INTERP_SPLINE, None, x.data_ptr(), y.data_ptr(), None, zi.data_ptr(),
                                     o[0].data_ptr(), o[1].data_ptr(), st.data_ptr(), q, s.cuda_stream)
            got[k] = (rc, *o, st)

        th = [threading.Thread(target=work, args=(k,)) for k in range(6)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        same = lambda a, b: bool(((a == b) | (torch.isnan(a) & torch.isnan(b))).all())  # noqa: E731
        for rc, out, der, st in got:
            assert rc == 0
            assert same(out, ref[0]) and same(der, ref[1]) and torch.equal(st, ref[2])
        want.close()
        shared.close()
