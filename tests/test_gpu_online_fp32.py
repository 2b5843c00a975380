"""The fp32 pass of the online solver (three bf16 parts, csrc/online.hip): the
paddings of d, ends of tiles and splits, and exponents past the range where
the potential's high part is a multiple of 2^-10; against the float64 oracle
and the float64 pass."""

import numpy as np
import pytest
import torch

import oracle.sinkhorn as osk
from pot_amd import online

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,d", [(1, 1, 1), (31, 33, 2), (128, 64, 16), (129, 65, 17),
                                   (300, 515, 3), (64, 700, 33), (257, 130, 100)])
@pytest.mark.parametrize("splits", [0, 3])
def test_fp32_pass_at_tile_edges(n, m, d, splits):
    rng = np.random.default_rng(n + m)
    x = rng.standard_normal((n, d)).astype(np.float32)
    y = (0.5 + rng.standard_normal((m, d))).astype(np.float32)
    a, b = rng.random(n) + 0.2, rng.random(m) + 0.2
    a, b = a / a.sum(), b / b.sum()
    x64, y64 = x.astype(np.float64), y.astype(np.float64)
    M = ((x64[:, None] - y64[None]) ** 2).sum(-1)
    M /= M.max()
    u, v, lg = online.sinkhorn_online(x, y, 0.05, a, b, numItermax=20, stopThr=0.0, warn=False,
                                      splits=splits)
    P = osk.sinkhorn_log(a, b, M, 0.05, numItermax=20, stopThr=0.0, warn=False)
    got = np.exp(-M / 0.05 + u.cpu().numpy()[:, None] + v.cpu().numpy()[None])
    mask = P >= 1e-30
    assert np.max(np.abs(got - P)[mask] / P[mask]) < 1e-5
    assert abs((got * M).sum() - (P * M).sum()) <= 1e-6 * (P * M).sum()


def test_fp32_pass_with_large_exponents():
    """Exponents of about 2^14 in base 2: an fp32 rounding of one is 2^-10, and
    a potential carries a few of them."""
    rng = np.random.default_rng(0)
    x = torch.tensor(3.0 * rng.standard_normal((200, 3)), dtype=torch.float32)
    y = torch.tensor(3.0 * rng.standard_normal((180, 3)), dtype=torch.float32)
    kw = dict(numItermax=1, stopThr=0.0, cost_scale=1.0, warn=False)
    u, v, _ = online.sinkhorn_online(x, y, 2e-3, **kw)
    u64, v64, _ = online.sinkhorn_online(x, y, 2e-3, precision="f64", **kw)
    assert v64.abs().max() > 1000  # natural units
    shift = (u - u64).mean()  # a common shift of u against v is free
    assert (u - u64 - shift).abs().max() < 16 * 2.0 ** -10
    assert (v - v64 + shift).abs().max() < 16 * 2.0 ** -10
