"""Split point-cloud problems whose parts wait for a workgroup."""

import numpy as np
import pytest
import torch

from pot_amd import ragged

pytestmark = pytest.mark.gpu


def test_a_part_waits_as_long_as_earlier_problems_take():
    """85 problems in three parts each and one more: its first part has the last
    CU, the others wait for the 1.5 million iterations (6.7 s) of the earlier
    problems, longer than parts at work wait for each other."""
    B = 86
    rng = np.random.default_rng(0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert 3 * (B - 1) < cus < 3 * B
    xs = [rng.standard_normal((96, 2)).astype(np.float32) for _ in range(B)]
    ys = [rng.standard_normal((64, 2)).astype(np.float32) for _ in range(B)]
    # (all points the same: solved in one iteration, without error)
    xs[-1] = ys[-1] = np.zeros((128, 2), np.float32)
    P = ragged.points_from_clouds(xs, ys, np.full(B, 0.5), normalize=False)
    res = ragged.sinkhorn_log_ragged_points(P, numItermax=1500000, stopThr=1e-13,
                                            order=np.arange(B), split=np.full(B, 3),
                                            unsolved="nan")
    assert (res.niter[:-1] == 1499999).all() and (res.status[:-1] == 1).all()
    assert res.status[-1].item() == 0 and res.niter[-1].item() == 0
    u, v = res.split(P, B - 1)
    np.testing.assert_allclose((u[:, None] + v[None]).cpu().numpy(), -2 * np.log(128), rtol=1e-6)


def _uneven(B):
    rng = np.random.default_rng(B)
    ns, ms = rng.integers(300, 512, B), rng.integers(300, 512, B)
    xs = torch.tensor(rng.standard_normal((ns.sum(), 4)), dtype=torch.float32, device="cuda")
    ys = torch.tensor(rng.standard_normal((ms.sum(), 4)), dtype=torch.float32, device="cuda")
    return ns, ms, xs, ys, np.exp(rng.uniform(np.log(0.02), np.log(0.1), B))


def test_a_split_solve_returns_without_a_wait():
    """unsolved="nan": work queued before the call is still running when it returns."""
    ns, ms, xs, ys, regs = _uneven(600)
    parts = ragged.auto_plan(ns, ms)
    assert parts.max() > 1
    P = ragged.points_from_clouds(list(xs.split(ns.tolist())), list(ys.split(ms.tolist())), regs)
    kw = dict(numItermax=20, stopThr=0.0, unsolved="nan", split=parts)
    want = ragged.sinkhorn_log_ragged_points(P, **kw)
    torch.cuda.synchronize()
    torch.cuda._sleep(50_000_000)
    before = torch.cuda.Event()
    before.record()
    got = ragged.sinkhorn_log_ragged_points(P, **kw)
    assert not before.query()
    torch.cuda.synchronize()
    assert torch.equal(got.u, want.u) and torch.equal(got.v, want.v)


def test_the_automatic_split_leaves_full_batches_whole():
    """More than two problems a CU: parts would only add work where the problems
    take about as many iterations each."""
    ns, ms, xs, ys, regs = _uneven(600)
    G = ragged.RaggedGraph(ns, ms, 4, numItermax=20, stopThr=0.0, cost="points")
    assert G.parts is None
    G = ragged.RaggedGraph(ns[:90], ms[:90], 4, numItermax=20, stopThr=0.0, cost="points")
    np.testing.assert_array_equal(G.parts, ragged.split_plan(ns[:90], ms[:90]))
