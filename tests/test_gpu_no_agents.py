"""Handles and scenarios without agents, in every layout: ticks run, readbacks
are empty, nothing is counted."""
import numpy as np
import pytest

import msim
from msim import scenarios as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("binning", [0, 1, 2, 3])
def test_simulation_without_agents(binning):
    sc = S.config(1, scale=0.1)
    g = msim.Simulation(sc.roads, sc.conns, sc.entities[:0], sc.pc, speed=sc.speed[:0], binning=binning, graph_ticks=4)
    for ticks in (1, 3, 11):
        g.run_ticks(ticks)
        assert g.entities().shape[0] == 0 and g.state()["pos"].shape == (0, 2) and g.cells().shape == (0, 2)
        assert g.pairs()[0] == 0 and not g.pairs()[1].any()
    g.dispatch()
    g.dispatch()
    g.sync()


@pytest.mark.parametrize("binning", [0, 2, 3])
def test_batch_with_empty_scenarios(binning):
    full = S.config(1, scale=0.05)
    empty = S.Scenario("empty", full.roads, full.conns, full.entities[:0], full.speed[:0], full.pc, 0, full.world)
    b = msim.Batch([empty, full, empty], binning=binning, graph_ticks=4)
    g = msim.Simulation(full.roads, full.conns, full.entities, full.pc, speed=full.speed)
    b.run_ticks(13)
    g.run_ticks(13)
    np.testing.assert_array_equal(b.state(1)["pos"].view(np.uint32), g.state()["pos"].view(np.uint32))
    assert b.state(0)["pos"].shape == (0, 2) and b.state(2)["rng"].shape == (0, 4)
    total, last = b.pairs()
    assert total.tolist() == [0, g.pairs()[0], 0] and last[0] == 0 and last[2] == 0
    b.sync()
