"""Crowds and sizes past which a path changes: a whole-world table kept or left
for the agents' own, windows of more agents than the sorted move's map can
index, more neighbour workgroups than fit the GPU at once; against the CPU
oracle bit for bit."""
import numpy as np
import pytest

import msim
from msim import scenarios as S
from test_gpu_parity import assert_same, pair
from test_gpu_tables import _world

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("agents,buckets", [(73_700, 1 << 12), (90_000, 1 << 17)])
@pytest.mark.parametrize("binning", [0, 1, 2, 3])
def test_crowded_world_of_one_table_or_the_other(agents, buckets, binning):
    """17 x 17 cells: a bucket per cell up to 8,192 agents per 512 buckets."""
    sc = _world(9, 9, agents, 16.0)
    g, o = pair(sc, threads=8, binning=binning, graph_ticks=2)
    info = g.info()
    assert info["table_width"] * info["table_height"] == buckets
    g.run_ticks(3)
    o.run_ticks(3)
    assert_same(g.state(), o.st, f"{agents} agents")
    assert g.pairs()[0] == o.pairs_total
    g.sync()


@pytest.mark.parametrize("width", [9, 5])  # lists of leavers; windows
def test_window_past_sixteen_bits(width):
    """Two segments of some 75,000 agents: moved and listed by the rank pass."""
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, 150_000, 11)
    g, o = pair(sc, threads=8, binning=3, graph_ticks=3, table_log2=13, segment_log2=12, table_width_log2=width)
    for ticks in (1, 8):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        assert_same(g.state(), o.st, f"rows of 2^{width}, {ticks} ticks")
    for _ in range(4):
        g.dispatch()
        o.dispatch()
    assert_same(g.state(), o.st, f"rows of 2^{width}, dispatches")
    assert g.pairs()[0] == o.pairs_total
    g.sync()


def test_batched_window_past_sixteen_bits():
    scs = [_world(9, 9, 70_000, 16.0), _world(9, 9, 300, 16.0)]
    b = msim.Batch(scs, binning=3, graph_ticks=3)
    b.run_ticks(5)
    for k, sc in enumerate(scs):
        g = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed, binning=0)
        g.run_ticks(5)
        x, y = b.state(k), g.state()
        for key in x:
            np.testing.assert_array_equal(np.ascontiguousarray(x[key]).view(np.uint32),
                                          np.ascontiguousarray(y[key]).view(np.uint32), err_msg=f"{key} of {k}")
    b.sync()


def test_more_workgroups_than_fit_at_once():
    """2,050 neighbour workgroups of two slots a lane and 1,024 segments, dealt
    to the XCDs in chunks, with a remainder."""
    n = (1 << 20) + 1_000
    sc = S.config(2, scale=0.3)
    sc.entities, sc.speed = S.place_agents(sc.roads, n, 4)
    g, o = pair(sc, threads=8, binning=3, graph_ticks=2)
    for ticks in (1, 3, 2):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        assert_same(g.state(), o.st, f"{ticks} ticks")
    assert g.pairs()[0] == o.pairs_total
    g.sync()
    b = msim.Batch([sc, S.config(1, scale=0.1)], binning=3, graph_ticks=2)
    b.run_ticks(6)
    x, y = b.state(0), g.state()
    for key in x:
        np.testing.assert_array_equal(np.ascontiguousarray(x[key]).view(np.uint32),
                                      np.ascontiguousarray(y[key]).view(np.uint32), err_msg=key)
    b.sync()
