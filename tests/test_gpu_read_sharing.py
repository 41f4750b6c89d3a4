"""Handles of one process share the pinned slots of their readbacks: many
handles one after the other and at once, read from several threads."""
import threading

import numpy as np
import pytest

import msim
from msim import scenarios as S

pytestmark = pytest.mark.gpu


def _simulation(n, binning):
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, n, n)
    g = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed, binning=binning)
    g.run_ticks(3)
    return g


@pytest.mark.parametrize("n", [500, 40_000, 600_000])
def test_first_and_later_reads_of_many_handles(n):
    want = None
    for kept in range(3):
        handles = [_simulation(n, 0) for _ in range(4)]
        for g in handles + handles:
            e, st = g.entities(), g.state()
            if want is None:
                want = e
            np.testing.assert_array_equal(e.view(np.uint8), want.view(np.uint8))
            np.testing.assert_array_equal(st["pos"].view(np.uint32), want["pos"].view(np.uint32))
        for g in handles:
            g.close()


def test_readers_in_several_threads():
    sizes = (500, 20_000, 45_000, 300_000)
    handles = [_simulation(n, b) for n, b in zip(sizes, (0, 3, 0, 3))]
    want = [(g.entities(), g.state()) for g in handles]
    failures = []

    def read(g, e, st):
        try:
            for _ in range(12):
                np.testing.assert_array_equal(g.entities().view(np.uint8), e.view(np.uint8))
                got = g.state()
                for k in st:
                    np.testing.assert_array_equal(np.ascontiguousarray(got[k]).view(np.uint32),
                                                  np.ascontiguousarray(st[k]).view(np.uint32), err_msg=k)
        except Exception as ex:  # reported by the test's own thread
            failures.append(ex)

    threads = [threading.Thread(target=read, args=(g, *w)) for g, w in zip(handles, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[0]
