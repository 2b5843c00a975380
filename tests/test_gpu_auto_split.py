"""The automatic split of point-cloud batches (ragged.auto_plan) with more parts
than the GPU has CUs, against one workgroup per problem.

After a fixed number of iterations the potentials differ by the order of the
float32 column sums: at most 2 x 512 x 2^-24 = 6e-5 in log units for each of
u and v (the iteration does not amplify them).
"""

import numpy as np
import pytest
import torch

from pot_amd import ragged

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,lo,hi", [(300, 400, 512), (90, 33, 512)])
def test_more_parts_than_cus(B, lo, hi):
    rng = np.random.default_rng(B)
    ns, ms = rng.integers(lo, hi + 1, B), rng.integers(lo, hi + 1, B)
    xs = [rng.standard_normal((n, 5)).astype(np.float32) for n in ns]
    ys = [(0.5 + rng.standard_normal((m, 5))).astype(np.float32) for m in ms]
    regs = np.exp(rng.uniform(np.log(0.02), np.log(0.1), B))
    parts = ragged.auto_plan(ns, ms)
    assert parts.sum() > (256 if B == 300 else B) and parts.max() > 1
    P = ragged.points_from_clouds(xs, ys, regs)
    one = ragged.sinkhorn_log_ragged_points(P, numItermax=15, stopThr=0.0, split=None)
    many = ragged.sinkhorn_log_ragged_points(P, numItermax=15, stopThr=0.0)
    torch.cuda.synchronize()
    assert torch.equal(one.status, many.status) and torch.equal(one.niter, many.niter)
    assert (one.u - many.u).abs().max().item() < 1.2e-4
    assert (one.v - many.v).abs().max().item() < 1.2e-4
    G = ragged.RaggedGraph(ns, ms, 5, numItermax=15, stopThr=0.0, cost="points")
    for _ in range(3):
        r = G.solve(xs, ys, regs)
        torch.cuda.synchronize()
        assert torch.equal(r.u, many.u) and torch.equal(r.v, many.v)
