"""Readbacks around the sizes where they change route: one pinned slot (2 MB in
all), one thread, several threads, pieces that do not fill a slot; partial
entity ranges and single arrays; plain and batched, both layouts."""
import ctypes

import numpy as np
import pytest

import msim
from msim import scenarios as S
from msim._lib import _ptr
from test_gpu_parity import assert_same, pair

pytestmark = pytest.mark.gpu


def _scenario(n):
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, n, n)
    return sc


# 48 bytes of state and 64 of entity per agent against 2^21-byte slots
@pytest.mark.parametrize("n", [1, 32768, 32769, 43690, 43691, 87383, 350001])
@pytest.mark.parametrize("binning", [0, 3])
def test_state_and_entities_match_oracle(n, binning):
    sc = _scenario(n)
    g, o = pair(sc, threads=4, binning=binning)
    g.run_ticks(3)
    o.run_ticks(3)
    assert_same(g.state(), o.st, f"{n} agents")
    g.dispatch()
    o.dispatch()
    st = g.state()
    assert_same(st, o.st, f"{n} agents after a move")
    e = g.entities()
    for field, key in (("pos", "pos"), ("target", "tgt"), ("direction", "dir"), ("roadIndex", "road"),
                       ("randomState", "rng")):
        np.testing.assert_array_equal(e[field].view(np.uint32), st[key].view(np.uint32), err_msg=field)
    for first, count in ((0, n), (n // 3, n - n // 3), (n - 1, 1)):
        np.testing.assert_array_equal(g.entities(first, count).view(np.uint8), e[first:first + count].view(np.uint8))
    road = np.zeros(n, np.uint32)
    g._check(g.lib.msim_read_state(g.h, None, None, None, _ptr(road), None, None))
    np.testing.assert_array_equal(road, st["road"])


@pytest.mark.parametrize("binning", [0, 3])
def test_batch_states_match_plain_runs(binning):
    scs = [_scenario(n) for n in (1, 43691, 5000, 90001)]
    b = msim.Batch(scs, binning=binning)
    b.run_ticks(4)
    for k, sc in enumerate(scs):
        g = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed)
        g.run_ticks(4)
        x, y = b.state(k), g.state()
        for key in x:
            np.testing.assert_array_equal(np.ascontiguousarray(x[key]).view(np.uint32),
                                          np.ascontiguousarray(y[key]).view(np.uint32), err_msg=f"{key} of {k}")
        nc = np.zeros(sc.entities.shape[0], np.uint32)
        b._check(b.lib.msim_batch_read_state(b.h, k, None, None, None, None, None, ctypes.c_void_p(nc.ctypes.data)))
        np.testing.assert_array_equal(nc, y["ncount"])
