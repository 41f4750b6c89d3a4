"""The segment tape the forward run leaves for the backward pass, the lists of
slots with neighbours, and the per-agent theta sums: gradients from the tape as
recorded, from a replay of every segment, and from runs that keep their
schedule agree; small, ragged and crowded agent sets, with and without
avoidance, against the binary64 host adjoint's tolerance."""
import numpy as np
import pytest
import torch

import msim
from msim import scenarios as S
from msim.adjoint import DiffRun

pytestmark = pytest.mark.gpu


def _scenarios(sizes, nodes=64, seed=21):
    out = []
    for k, n in enumerate(sizes):
        sc = S.adjoint_config(1, agents=max(n, 1), nodes=nodes, seed=seed + k)[0]
        sc.entities, sc.speed = sc.entities[:n], sc.speed[:n]
        out.append(sc)
    return out


def _gradients(run, theta, alpha, g, times=1, between=None):
    t = theta.clone().requires_grad_(True)
    a = alpha.clone().requires_grad_(True)
    pos = run(t, a)
    if between is not None:
        between(run, theta)
    out = []
    for k in range(times):
        gt, ga = torch.autograd.grad(pos, (t, a), g, retain_graph=k + 1 < times)
        out.append((gt.double().cpu().numpy(), float(ga)))
    return pos.detach().cpu().numpy(), out


# sums of the same binary64 terms in another order, rounded to binary32
def _close(x, y):
    scale = np.abs(x[0]).max()
    np.testing.assert_allclose(x[0], y[0], rtol=0, atol=2.0 ** -22 * scale)
    assert abs(x[1] - y[1]) <= 2.0 ** -22 * max(abs(x[1]), abs(y[1])) + 1e-12 * scale


@pytest.mark.parametrize("sizes", [(1,), (63, 0, 65), (256, 129), (1500, 900)])
@pytest.mark.parametrize("ticks,every", [(7, 7), (7, 50), (23, 10), (20, 10), (9, 1)])
@pytest.mark.parametrize("alpha", [0.0, 0.03])
@pytest.mark.parametrize("arrivals", ["frozen", "carry"])
def test_taped_and_replayed_gradients_agree(sizes, ticks, every, alpha, arrivals):
    scs = _scenarios(sizes)
    rng = torch.Generator().manual_seed(3)
    n_roads = sum(sc.roads.shape[0] for sc in scs)
    theta = torch.exp(0.2 * torch.randn(n_roads, generator=rng)).cuda()
    al = torch.tensor(alpha).cuda()
    n = sum(sizes)
    g = torch.randn(n, 2, generator=rng).cuda()
    b = msim.Batch(scs)
    run = DiffRun(b, ticks, checkpoint_every=every, arrival_gradient=arrivals)
    pos, (taped, replayed) = _gradients(run, theta, al, g, times=2)
    b2 = msim.Batch(scs)
    kept = DiffRun(b2, ticks, checkpoint_every=every, keep_schedule=True, arrival_gradient=arrivals)
    # a replay between the runs leaves the working state elsewhere
    pos2, (schedule,) = _gradients(kept, theta, al, g, between=lambda r, th: r.replay(th * 1.01, alpha))
    np.testing.assert_array_equal(pos.view(np.uint32), pos2.view(np.uint32))
    _close(taped, replayed)
    _close(taped, schedule)
    assert np.isfinite(taped[0]).all() and np.abs(taped[0]).max() > 0.0
    pos3, (again,) = _gradients(run, theta, al, g)
    np.testing.assert_array_equal(pos.view(np.uint32), pos3.view(np.uint32))
    _close(taped, again)
    b.close()
    b2.close()


# one launch copies a snapshot's arrays: short arrays, word remainders, and
# arrays longer than one pass of the copying grid (2^22 words)
@pytest.mark.parametrize("sizes,nodes", [((1,), 64), ((3,), 64), ((5, 2), 64), ((1_048_577, 31), 20_000)])
@pytest.mark.parametrize("uniform", [False, True])
def test_runs_start_again_from_the_initial_state(sizes, nodes, uniform):
    scs = _scenarios(sizes, nodes=nodes)
    if uniform:
        for sc in scs:
            sc.speed = None
    n = sum(sizes)
    b, ref = msim.Batch(scs), msim.Batch(scs)
    ref.run_ticks(4)
    expect = np.concatenate([ref.state(k)["pos"] for k in range(len(scs))])
    run = DiffRun(b, 4, checkpoint_every=2)
    theta = torch.ones(b.n_roads, device="cuda")
    g = torch.ones(n, 2, device="cuda")
    grads = []
    for _ in range(3):
        pos, (taped, replayed) = _gradients(run, theta, torch.tensor(0.0).cuda(), g, times=2)
        np.testing.assert_array_equal(pos.view(np.uint32), expect.view(np.uint32))
        _close(taped, replayed)
        grads.append(taped)
    _close(grads[0], grads[2])
    b.close()
    ref.close()


# the multipliers are checked on the device, in 2^17 threads: few of them, and
# more than one pass; the largest (its agents cross many cells a tick, and the
# rebinning windows have to allow for that) and a bad one at the end
@pytest.mark.parametrize("sizes,nodes", [((40,), 64), ((3000, 500), 90_000)])
@pytest.mark.parametrize("bad", [-1.0, float("inf"), float("nan")])
def test_multipliers_are_checked_on_the_device(sizes, nodes, bad):
    scs = _scenarios(sizes, nodes=nodes)
    b = msim.Batch(scs)
    run = DiffRun(b, 6, checkpoint_every=3)
    theta = torch.ones(b.n_roads, device="cuda")
    theta[b.n_roads // 2 :] = 9.0
    theta[-1] = 20.0
    al = torch.tensor(0.01).cuda()
    g = torch.ones(sum(sizes), 2, device="cuda")
    pos, (expect,) = _gradients(run, theta, al, g)
    out = torch.empty(sum(sizes), 2, device="cuda")
    # elsewhere in an allocation, and pinned memory of the host
    held = torch.cat([torch.zeros(3, device="cuda"), theta])
    host = torch.empty(b.n_roads, pin_memory=True).copy_(theta)
    for ptr in (held[3:].data_ptr(), host.data_ptr()):
        torch.cuda.synchronize()
        b.diff_forward(ptr, 0.01, out.data_ptr())
        np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), pos.view(np.uint32))
    wrong = theta.clone()
    wrong[-1] = bad
    t = theta.clone().requires_grad_(True)
    a = al.clone().requires_grad_(True)
    p = run(t, a)
    torch.cuda.synchronize()
    for _ in range(2):
        with pytest.raises(msim.MsimError, match=rf"theta\[{b.n_roads - 1}\]"):
            b.diff_forward(wrong.data_ptr(), 0.01, out.data_ptr())
    gt, ga = torch.autograd.grad(p, (t, a), g)  # the run before is still there
    _close(expect, (gt.double().cpu().numpy(), float(ga)))
    b.close()


# a tick of the adjoint takes 4, 8 or 16 groups of 64 slots a workgroup
@pytest.mark.parametrize("agents", [326_980, 326_981, 654_660, 654_661])
def test_group_counts_of_the_adjoint_agree(agents):
    scs = _scenarios((agents, 700), nodes=40_000)
    alone = _scenarios((1, 700), nodes=40_000)[1:]
    # the second scenario alone runs with the smallest count
    grads = []
    for maps in (scs, alone):
        b = msim.Batch(maps)
        n, first = sum(sc.entities.shape[0] for sc in maps), b.n_roads - maps[-1].roads.shape[0]
        g = torch.zeros(n, 2, device="cuda")
        g[-700:] = torch.randn(700, 2, generator=torch.Generator().manual_seed(9)).cuda()
        theta = torch.ones(b.n_roads, device="cuda")
        _, (got,) = _gradients(DiffRun(b, 8, checkpoint_every=4), theta, torch.tensor(0.03).cuda(), g)
        assert not got[0][:first].any()
        grads.append((got[0][first:], got[1]))
        b.close()
    _close(grads[1], grads[0])
