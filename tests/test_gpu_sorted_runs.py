"""Ticks inside runs, whose launches differ from single dispatches': the sorted
state's two-launch tick, the one-launch scan of small tables, and statistics
folded by the next move, at the sizes where their workgroup dealing can go
wrong, against the CPU oracle bit for bit."""
import numpy as np
import pytest

import msim
import orc
from msim import scenarios as S
from test_gpu_parity import assert_same, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("agents", [1, 64, 511, 513, 5000])
@pytest.mark.parametrize("opts", [dict(table_log2=12), dict(table_log2=12, segment_log2=9),
                                  dict(table_log2=19, segment_log2=9), dict(segment_log2=10, graph_ticks=7)])
def test_run_matches_oracle(agents, opts):
    """More route than neighbour workgroups and the reverse, counts that are
    no multiple of eight, one segment and many, direct and captured ticks."""
    sc = S.config(1, scale=0.5)
    sc.entities, sc.speed = sc.entities[:agents], sc.speed[:agents]
    g, o = pair(sc, binning=3, **opts)
    for ticks in (1, 45, 2, 33):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        assert_same(g.state(), o.st, f"{agents} agents, {opts}")
    total, hist = g.pairs()
    assert total == o.pairs_total
    assert hist.tolist() == o.pair_hist
    g.sync()


@pytest.mark.parametrize("n_scen", [1, 8, 63, 65])
def test_batch_run_folds_every_scenarios_pairs(n_scen):
    """Pair totals and the last tick's pairs of every scenario, the earlier
    ticks' totals folded by the moves that follow them."""
    scs = S.batch_config(n_scen, scale=0.004, seed=11)
    b = msim.Batch(scs, binning=3, graph_ticks=6)
    b.run_ticks(31)
    tot, last = b.pairs()
    for s, sc in enumerate(scs):
        o = orc.OracleSim(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed)
        o.run_ticks(31)
        assert int(tot[s]) == o.pairs_total and int(last[s]) == o.pair_hist[-1], f"scenario {s}"
        st = b.state(s)
        np.testing.assert_array_equal(st["pos"].view(np.uint32), o.st.pos.view(np.uint32), err_msg=f"scenario {s}")
        np.testing.assert_array_equal(st["rng"], o.st.rng, err_msg=f"scenario {s}")
    b.sync()


@pytest.mark.parametrize("opts,agents", [
    (dict(table_log2=12, segment_log2=12, table_width_log2=8), 4000),   # one segment: nothing leaves it
    (dict(table_log2=12, segment_log2=11, table_width_log2=7), 4000),   # two: each is above and below the other
    (dict(table_log2=12, segment_log2=10, table_width_log2=6), 4000),   # four, a few rows each
    (dict(table_log2=13, segment_log2=9, table_width_log2=7), 4000),    # margin wider than 3/4 of a segment
    (dict(table_log2=14, segment_log2=12, table_width_log2=10), 60000),  # more leavers than their slots fit in LDS
    (dict(table_log2=13, segment_log2=12, table_width_log2=9), 60000),  # crowded past the map and its 16-bit window
    (dict(table_log2=18, segment_log2=10, table_width_log2=7), 20000),  # 256 segments: workgroups of 1,024 threads
    (dict(table_log2=19, segment_log2=10, table_width_log2=7), 20000),  # 512: of 512
])
def test_lists_of_leaving_agents_match_oracle(opts, agents):
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, agents, 5)
    g, o = pair(sc, threads=4, binning=3, graph_ticks=6, **opts)
    for ticks in (1, 20):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        assert_same(g.state(), o.st, f"{opts}")
    for _ in range(6):  # the same lists through single dispatches
        g.dispatch()
        o.dispatch()
    assert_same(g.state(), o.st, f"{opts}, dispatches")
    assert g.pairs()[0] == o.pairs_total
    g.sync()


@pytest.mark.parametrize("agents", [1, 257, 1025, 5000])
@pytest.mark.parametrize("opts", [dict(binning=0), dict(binning=0, route_queue=1), dict(binning=1),
                                  dict(binning=1, route_queue=1, table_log2=15), dict(binning=1, table_log2=16),
                                  dict(binning=2, collide_mode=1), dict(binning=3, collide_mode=2)])
def test_run_statistics_match_oracle(agents, opts):
    """Pair history, insertions and state after direct and captured ticks, with
    renumberings in between, in every layout."""
    sc = S.config(1, scale=0.5)
    sc.entities, sc.speed = sc.entities[:agents], sc.speed[:agents]
    g, o = pair(sc, graph_ticks=6, reorder_interval=3, **opts)
    ref = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed)
    for ticks in (1, 5, 26, 2, 13):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        for _ in range(ticks):
            ref.sim_tick()
        assert_same(g.state(), o.st, f"{agents} agents, {opts}")
        np.testing.assert_array_equal(g.debug_data(), ref.debug_data())
    total, hist = g.pairs()
    assert total == o.pairs_total
    assert hist.tolist() == o.pair_hist
    g.sync()


@pytest.mark.parametrize("n_scen", [1, 31, 33])
@pytest.mark.parametrize("binning", [0, 2])
def test_classic_batch_run_folds_every_scenarios_pairs(n_scen, binning):
    scs = S.batch_config(n_scen, scale=0.004, seed=12)
    b = msim.Batch(scs, binning=binning, graph_ticks=6, reorder_interval=3)
    b.run_ticks(29)
    tot, last = b.pairs()
    for s, sc in enumerate(scs):
        o = orc.OracleSim(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed)
        o.run_ticks(29)
        assert int(tot[s]) == o.pairs_total and int(last[s]) == o.pair_hist[-1], f"scenario {s}"
    b.sync()
