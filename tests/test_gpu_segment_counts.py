"""The sorted state's counts per segment and per group of segments, at the
sizes where the groups change: one group, a last one that is not full, groups
of 16 to 128 segments, scenarios that share a group; with lists of leavers and
with windows, in two-launch and single-dispatch ticks, against the CPU oracle
bit for bit."""
import numpy as np
import pytest

import msim
import orc
from msim import scenarios as S
from test_gpu_parity import assert_same, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("table,seg,width", [
    (12, 9, 6),    # 8 segments: half a group
    (13, 9, 5),    # 16
    (17, 9, 9),    # 256, windows of seven segments
    (18, 9, 7),    # 512
    (19, 9, 7),    # 1,024: groups of 32
    (19, 9, 9),
    (24, 9, 7),    # 32,768: groups of 128
])
@pytest.mark.parametrize("mode", [0, 1])
def test_segment_counts_match_oracle(table, seg, width, mode):
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, 20_000, table)
    g, o = pair(sc, threads=4, binning=3, graph_ticks=6, table_log2=table, segment_log2=seg, table_width_log2=width,
                collide_mode=mode)
    for ticks in (1, 17, 2):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        assert_same(g.state(), o.st, f"2^{table} buckets, 2^{seg} a segment, rows of 2^{width}")
    for _ in range(4):  # the same counts through single dispatches
        g.dispatch()
        o.dispatch()
    assert_same(g.state(), o.st, "dispatches")
    assert g.pairs()[0] == o.pairs_total
    g.sync()


@pytest.mark.parametrize("n_scen,segment", [(1, 9), (3, 9), (70, 9), (70, 11)])
def test_scenarios_sharing_groups_match_oracle(n_scen, segment):
    scs = S.batch_config(n_scen, scale=0.01, seed=7)
    b = msim.Batch(scs, binning=3, graph_ticks=6, segment_log2=segment)
    b.run_ticks(20)
    tot, last = b.pairs()
    for s, sc in enumerate(scs):
        o = orc.OracleSim(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed)
        o.run_ticks(20)
        assert int(tot[s]) == o.pairs_total and int(last[s]) == o.pair_hist[-1], f"scenario {s}"
        st = b.state(s)
        np.testing.assert_array_equal(st["pos"].view(np.uint32), o.st.pos.view(np.uint32), err_msg=f"scenario {s}")
        np.testing.assert_array_equal(st["rng"], o.st.rng, err_msg=f"scenario {s}")
    b.sync()
