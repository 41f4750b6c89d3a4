"""Readbacks into memory that the caller has pinned and into device memory, at
sizes within one slot and past it; plain and batched, both layouts."""
import ctypes

import numpy as np
import pytest
import torch

import msim
from msim import scenarios as S

pytestmark = pytest.mark.gpu


def _memory(kind, nbytes, offset=0):
    """(pointer, function giving the bytes as numpy, keeper) of zeroed memory."""
    if kind == "device":
        t = torch.zeros(nbytes + offset, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
    else:
        t = torch.zeros(nbytes + offset, dtype=torch.uint8, pin_memory=kind == "pinned")
    return ctypes.c_void_p(t.data_ptr() + offset), lambda: t.cpu().numpy()[offset:]


def _scenario(n):
    sc = S.config(1)
    sc.entities, sc.speed = S.place_agents(sc.roads, n, n)
    return sc


@pytest.mark.parametrize("kind", ["pinned", "device", "pageable"])
@pytest.mark.parametrize("n,binning", [(1, 0), (5000, 3), (32769, 0), (150001, 3)])
def test_entities_cells_and_state(kind, n, binning):
    sc = _scenario(n)
    g = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed, binning=binning)
    g.run_ticks(4)
    want, cells, state = g.entities().view(np.uint8).reshape(-1), g.cells(), g.state()
    for offset in (0, 64):
        p, got = _memory(kind, 64 * n, offset)
        g._check(g.lib.msim_read_entities(g.h, p, 0, n))
        np.testing.assert_array_equal(got(), want)
    p, got = _memory(kind, 8 * n)
    g._check(g.lib.msim_read_cells(g.h, p))
    np.testing.assert_array_equal(got().view(np.int32), cells.reshape(-1))
    if kind == "device":  # states go to host memory
        return
    parts = [_memory(kind, state[k].nbytes) for k in ("pos", "tgt", "dir", "road", "rng", "ncount")]
    g._check(g.lib.msim_read_state(g.h, *(p for p, _ in parts)))
    for (_, got), key in zip(parts, ("pos", "tgt", "dir", "road", "rng", "ncount")):
        np.testing.assert_array_equal(got(), np.ascontiguousarray(state[key]).view(np.uint8).reshape(-1), err_msg=key)


@pytest.mark.parametrize("kind", ["pinned", "device"])
def test_batch(kind):
    scs = [_scenario(n) for n in (5000, 90001)]
    b = msim.Batch(scs, binning=3)
    b.run_ticks(4)
    total, last = b.pairs()
    p, got = _memory(kind, 16)
    q, got_last = _memory(kind, 8)
    b._check(b.lib.msim_batch_read_pairs(b.h, p, q))
    np.testing.assert_array_equal(got().view(np.uint64), total)
    np.testing.assert_array_equal(got_last().view(np.uint32), last)
    for k in range(2 if kind == "pinned" else 0):
        st = b.state(k)
        p, got = _memory(kind, st["pos"].nbytes)
        r, got_rng = _memory(kind, st["rng"].nbytes)
        b._check(b.lib.msim_batch_read_state(b.h, k, p, None, None, None, r, None))
        np.testing.assert_array_equal(got(), np.ascontiguousarray(st["pos"]).view(np.uint8).reshape(-1))
        np.testing.assert_array_equal(got_rng(), np.ascontiguousarray(st["rng"]).view(np.uint8).reshape(-1))
