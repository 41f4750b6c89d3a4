"""Insertions, pair totals and the pair history, at capacities of the history
from one entry to one whose readback takes several slots, before and after it
wraps round; against the CPU oracle."""
import ctypes

import numpy as np
import pytest

from msim import scenarios as S
from msim._lib import _ptr
from test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [1, 2, 4, 16, 4096, 1 << 20])
@pytest.mark.parametrize("binning", [0, 3])
def test_counters_match_oracle(capacity, binning):
    sc = S.config(1, scale=0.3)
    g, o = pair(sc, binning=binning, history_capacity=capacity, graph_ticks=4)
    for ticks in (1, 2, 21, 1):
        g.run_ticks(ticks)
        o.run_ticks(ticks)
        for _ in range(2):  # without and with pinned memory
            for n in (4096, 3, 1, 0):
                total, hist = g.pairs(n)
                assert total == o.pairs_total
                assert hist.tolist() == o.pair_hist[len(o.pair_hist) - min(n, capacity, len(o.pair_hist)):]
            total, got = np.zeros(1, np.uint64), ctypes.c_uint32(9)
            g._check(g.lib.msim_read_pairs(g.h, _ptr(total), None, 5, ctypes.byref(got)))
            assert int(total[0]) == o.pairs_total and got.value == 0
            debug = g.debug_data()
            assert debug[1] == o.pairs_total % 2 ** 32 and debug[2:].max() == 0
        assert debug[0] >= sc.entities.shape[0]
    g.sync()
