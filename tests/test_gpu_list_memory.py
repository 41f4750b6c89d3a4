"""The sorted state's lists of leavers take no memory of their own per agent,
and leave every readback what it is (they lie in the binned positions)."""
import numpy as np
import pytest

import msim
from msim import scenarios as S
from test_gpu_parity import assert_same, pair

pytestmark = pytest.mark.gpu


def test_lists_take_no_memory_per_agent():
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, 50_000, 3)
    # rows of 2^5: margins too small for lists; rows of 2^8: lists (both 64 segments)
    plain, lists = (msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed, binning=3, table_log2=16,
                                    segment_log2=10, table_width_log2=w).info()["device_bytes"] for w in (5, 8))
    assert lists - plain < 50_000


def test_readbacks_between_moves():
    sc = S.config(1)
    g, o = pair(sc, binning=3, graph_ticks=4, table_log2=16, segment_log2=10, table_width_log2=8)
    for ticks in (1, 1, 9):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        cells = g.cells()
        np.testing.assert_array_equal(cells, np.floor(o.st.pos / g.info()["cell_size"]).astype(np.int32))
        xy, counts, total = g.grid_occupancy()
        want, n = np.unique(cells, axis=0, return_counts=True)
        at = np.lexsort((xy[:, 1], xy[:, 0]))
        assert total == want.shape[0]
        np.testing.assert_array_equal(xy[at], want)
        np.testing.assert_array_equal(counts[at], n)
        g.entities()
        assert_same(g.state(), o.st, f"{ticks} ticks")
    g.sync()
