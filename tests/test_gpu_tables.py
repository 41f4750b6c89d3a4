"""Automatic bucket tables: worlds that fit one bucket per cell, worlds just
past that, one-cell and one-row worlds, crowded small worlds; every layout
against the CPU oracle bit for bit."""
import numpy as np
import pytest

import msim
from msim import scenarios as S
from test_gpu_parity import assert_same, pair

pytestmark = pytest.mark.gpu


def _world(nodes_x, nodes_y, n, radius, spacing=32.0):
    x, y = np.meshgrid(np.arange(nodes_x), np.arange(nodes_y))
    xy = np.stack([x.ravel() * spacing - 40.0, y.ravel() * spacing - 7.0], axis=1).astype(np.float32)
    idx = np.arange(nodes_x * nodes_y).reshape(nodes_y, nodes_x)
    edges = np.concatenate([np.stack([idx[:, :-1].ravel(), idx[:, 1:].ravel()], 1),
                            np.stack([idx[:-1].ravel(), idx[1:].ravel()], 1)])
    roads, conns = S.build_roads(xy, edges)
    ents, speed = S.place_agents(roads, n, nodes_x + n)
    w, h = nodes_x * spacing, nodes_y * spacing
    return S.Scenario("grid", roads, conns, ents, speed, msim.push_consts(w, h, radius), 0, (w, h))


WORLDS = [(2, 1, 300, 64.0),     # one row of two cells
          (30, 1, 2000, 2.0),    # one road long, a row high
          (1, 30, 2000, 2.0),    # the same upright
          (32, 32, 9000, 16.0),  # 64 x 64 cells
          (33, 32, 9000, 16.0),  # a column more
          (9, 9, 70000, 16.0),   # crowded: the agents' own table
          (32, 64, 3000, 1.0)]   # folded


@pytest.mark.parametrize("world", WORLDS)
@pytest.mark.parametrize("binning", [0, 1, 2, 3])
def test_automatic_table_matches_oracle(world, binning):
    sc = _world(*world)
    g, o = pair(sc, threads=4, binning=binning, graph_ticks=8)
    g.run_ticks(19)
    o.run_ticks(19)
    assert_same(g.state(), o.st, f"{world}, binning {binning}")
    assert g.pairs()[0] == o.pairs_total
    g.sync()


@pytest.mark.parametrize("binning", [0, 2, 3])
def test_automatic_tables_of_a_batch_equal_plain_runs(binning):
    scs = [_world(nx, ny, n, 16.0) for nx, ny, n in ((32, 32, 9000), (2, 1, 40), (9, 9, 30000), (40, 3, 700))]
    b = msim.Batch(scs, binning=binning, graph_ticks=8)
    b.run_ticks(19)
    for k, sc in enumerate(scs):
        g = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed)
        g.run_ticks(19)
        x, y = b.state(k), g.state()
        for key in x:
            np.testing.assert_array_equal(np.ascontiguousarray(x[key]).view(np.uint32),
                                          np.ascontiguousarray(y[key]).view(np.uint32), err_msg=f"{key} of {k}")
    b.sync()
