"""Network-seeded inversions of more zones than one block a CU holds (65,536), whose kernels
read the network's operands from LDS: bit for bit the smaller calls' (operands in registers)
and the oracle's, on a batch whose last block is short, with blocks in which every, one or no
zone asks for the network."""
import ctypes

import numpy as np
import pytest

import harm_cool_amd as hc
from oracle_lib import _ptr, lib as olib
from test_gpu_stress import _host, _torch, _zone

pytestmark = pytest.mark.gpu
NARROW = 1 << 16
N = NARROW + 301
TAU = 1e-3


def _net(spec):
    tr = hc.stress_batch(NARROW, hc.stress_spec(0, seed=(777, 888, 999, 1111)))
    p = tr["guess"].clone()
    ret, _, _ = hc.utoprim2d_batch(tr["U"], tr["gcov"], tr["gcon"], tr["gdet"], p, spec.gam)
    feat, targ, valid = hc.mlp_pairs(tr["U"], tr["gcov"], tr["gcon"], tr["gdet"], p, ret, spec.gam)
    m = hc.Mlp(seed=5)
    m.fit_norm(feat, targ, valid)
    m.set_loss_weights(1.0, 0.0)
    m.train(feat, targ, valid, batch=8192, steps=300, lr0=3e-3, lr1=2e-4)
    return m


@pytest.mark.parametrize("gate", [0.0, TAU])
def test_large_batch_equals_small_ones_and_the_oracle(gate):
    torch = _torch()
    spec = hc.stress_spec(0)
    m = _net(spec)
    b = hc.stress_batch(N, spec)
    # blocks of 256 zones: all poor starts, all exact ones (no first step above TAU), one
    # poor start among exact ones
    z = torch.arange(N, device="cuda:0")
    kind = (z // 256) % 3
    poor = (kind == 0) | ((kind == 2) & (z % 256 == 77))
    guess = torch.where(poor[None], b["guess"], b["prim_true"])

    def run(sl):
        a = [b[k][..., sl].contiguous() for k in ("U", "gcov", "gcon", "gdet")]
        prim = guess[:, sl].clone(memory_format=torch.contiguous_format)
        return [*hc.utoprim2d_batch(*a, prim, spec.gam, mlp=m, gate=gate), prim]

    wide = run(slice(0, N))
    for sl in (slice(0, NARROW), slice(NARROW, N), slice(12345, 12345 + 5001)):
        for x, y in zip(wide, run(sl)):
            assert torch.equal(x[..., sl], y)
    _, W0, v0 = m.seed(b["U"], b["gcov"], b["gcon"], b["gdet"])
    torch.cuda.synchronize()
    h = _host(b)
    W0, v0, g0 = W0.cpu().numpy(), v0.cpu().numpy(), guess.cpu().numpy()
    ret, it, kc, prim = (t.cpu().numpy() for t in wide)
    L = olib()
    dp, ip = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)
    dbl = ctypes.c_double
    L.orc_utoprim_2d_learned.argtypes = [dp, dp, dp, dbl, dp, dbl, dbl, dbl, ctypes.c_int, ip, ip, ip]
    L.orc_utoprim_2d_gated.argtypes = [dp, dp, dp, dbl, dp, dbl, dbl, dbl, ctypes.c_int, dbl, ip, ip, ip]
    seeded = {True: 0, False: 0}
    pick = np.concatenate([np.random.default_rng(6).choice(N, 900, replace=False), np.arange(77 + 512, N, 768 * 4),
                           np.arange(N - 60, N)])
    for z in pick:
        U, gc, gn, gd = _zone(h, z)
        p = np.ascontiguousarray(g0[:, z].copy())
        ni, kz, s = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
        args = (_ptr(U), _ptr(gc), _ptr(gn), gd, _ptr(p), spec.gam, float(W0[z]), float(v0[z]), 1)
        tail = (ctypes.byref(ni), ctypes.byref(kz), ctypes.byref(s))
        r = L.orc_utoprim_2d_gated(*args, gate, *tail) if gate else L.orc_utoprim_2d_learned(*args, *tail)
        assert (np.int8(r), ni.value, kz.value) == (ret[z], it[z], kc[z]), z
        assert np.array_equal(p, prim[:, z]), z
        seeded[bool(poor[z])] += s.value
    if gate:
        assert seeded[True] > 300 and seeded[False] == 0, seeded
    m.close()
