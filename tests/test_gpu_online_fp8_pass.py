"""The two compilations of the fp8 pass of more than 96 coordinates (at most two
workgroups a CU, and more) and the merge of many splits."""

import pytest
import torch

from pot_amd import online

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [97, 128])
def test_potentials_do_not_depend_on_the_other_points(d):
    """One column update: a point's potential, less its log weight, is the same
    among 300 points (three workgroups) and among 66000 (516), bit for bit but for
    one rounding of the potential and one of the subtraction (5e-15 at 20)."""
    g = torch.Generator("cuda").manual_seed(d)
    X = torch.randn(200, d, generator=g, device="cuda")
    Y = torch.randn(66000, d, generator=g, device="cuda")
    kw = dict(numItermax=1, stopThr=0.0, precision="fp8", cost_scale=2.0 * d, splits=1, warn=False)
    few = online.sinkhorn_online(X, Y[:300], 0.1, **kw)[1] + torch.log(torch.tensor(300.0).double())
    many = online.sinkhorn_online(X, Y, 0.1, **kw)[1] + torch.log(torch.tensor(66000.0).double())
    assert (few - many[:300]).abs().max().item() < 5e-15


@pytest.mark.parametrize("precision", ["f32", "bf16", "f64"])
@pytest.mark.parametrize("splits", [2, 15, 16, 17, 33, 64])
def test_merge_of_splits(precision, splits):
    """As many splits as asked for (up to 64 of 64 points) and one: sums of float32
    terms in another order, 16 of them a tile (1e-6; float64 1e-12)."""
    g = torch.Generator("cuda").manual_seed(splits)
    X = torch.randn(150, 20, generator=g, device="cuda")
    Y = torch.randn(4096, 20, generator=g, device="cuda")
    kw = dict(numItermax=3, stopThr=0.0, precision=precision, cost_scale=40.0, warn=False)
    u1, v1, _ = online.sinkhorn_online(X, Y, 0.1, splits=1, **kw)
    u, v, _ = online.sinkhorn_online(X, Y, 0.1, splits=splits, **kw)
    tol = 1e-12 if precision == "f64" else 1e-6
    assert (u - u1).abs().max().item() < tol and (v - v1).abs().max().item() < tol
