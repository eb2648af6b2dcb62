"""Grids at the edges of the step's launch shapes, against the oracle: every direction's
fluxes in one launch (rows that fill no wavefront, two dimensions), the EMFs formed in the update there, and a step's end that adds more
phi planes than a block has threads."""
import pytest

import ceos_cases as cc
import test_gpu_ceos as tc
from harm_cool_amd.params import torus_params
from test_gpu_parity import _pair, assert_state_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2,n3,kw", [
    (10, 8, 1, {}), (33, 18, 1, dict(lim=3)), (12, 10, 38, {}), (11, 14, 6, dict(lim=3)),
    (13, 8, 30, dict(lim=1, hllf=0.0, laxf=1.0)), (8, 8, 320, {}),
])
def test_steps_match_oracle_at_launch_edges(n1, n2, n3, kw):
    g, o = _pair(torus_params(n1, n2, n3, **kw))
    g.init()
    assert o.init_torus() == 0
    for s in range(4):
        g.step_ch(1)
        assert o.step() == 0
        assert_state_close(g, o, f"step {s}")
        assert g.counters() == o.counters()
        assert g.time() == o.time()
    g.close()


@pytest.mark.parametrize("n1,n2,n3", [(10, 9, 40), (9, 10, 96), (12, 8, 38), (8, 8, 128)])
def test_cache_eos_rows_padded_to_wavefronts(n1, n2, n3):
    """phi rows of 63% (padded, idle lanes), 75%, 59% (not padded) and all of their
    wavefronts, one cache per radius."""
    g, o, caches = tc._pair(torus_params(n1, n2, n3), lambda P: cc.gas_rad(n=P.n1 + 4))
    g.init()
    assert o.init_torus() == 0
    for s in range(2):
        g.step_ch(1)
        assert o.step() == 0
        tc._same(g, o, f"step {s}")
    g.close()
    for c in caches:
        c.close()
