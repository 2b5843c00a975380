"""Forms of the inputs of solve_gromov_batch: transposed views, a reg per problem."""

import numpy as np
import pytest
import torch

from pot_amd import batch as pb

pytestmark = pytest.mark.gpu

B, N, M_ = 3, 9, 11


def _inputs(dtype):
    rng = np.random.default_rng(31)
    d = dict(dtype=dtype, device="cuda")
    C1 = torch.tensor(rng.random((B, N, N)), **d)
    C2 = torch.tensor(rng.random((B, M_, M_)), **d)
    T = torch.tensor(rng.random((B, N, M_)), **d)
    return C1, C2, T / T.sum((1, 2), keepdim=True), torch.tensor(rng.random((B, N, M_)), **d)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_transposed_start_and_cost(dtype):
    """A start or a cost held the other way round (the plan of the swapped
    problem) gives the bits of its contiguous copy."""
    C1, C2, T, M = _inputs(dtype)
    kw = dict(reg=0.1, max_iter=4, tol=0.0)
    want = pb.solve_gromov_batch(C1, C2, T_init=T, M=M, alpha=0.3, **kw)
    for k in range(3):
        t = T.transpose(1, 2).contiguous().transpose(1, 2) if k != 1 else T
        c = M.transpose(1, 2).contiguous().transpose(1, 2) if k != 0 else M
        assert not (t.is_contiguous() and c.is_contiguous())
        got = pb.solve_gromov_batch(C1, C2, T_init=t, M=c, alpha=0.3, **kw)
        assert torch.equal(got.plan, want.plan)
        assert torch.equal(got.potentials[0], want.potentials[0])
    t = T.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(pb.solve_gromov_batch(C1, C2, T_init=t, **kw).plan,
                       pb.solve_gromov_batch(C1, C2, T_init=T, **kw).plan)


def test_reg_per_problem():
    """Without the joint stops, each problem of a batch with its own reg is the
    lone problem at that reg (a few roundings apart, amplified by exponents up
    to 2 / 0.05: 1e-11)."""
    C1, C2, T, M = _inputs(torch.float64)
    regs = torch.tensor([0.05, 0.1, 0.2], dtype=torch.float64, device="cuda")
    kw = dict(max_iter=5, tol=0.0, max_iter_inner=30, tol_inner=0.0, alpha=0.4)
    got = pb.solve_gromov_batch(C1, C2, reg=regs[:, None, None], T_init=T, M=M, **kw)
    for p in range(B):
        s = slice(p, p + 1)
        one = pb.solve_gromov_batch(C1[s], C2[s], reg=float(regs[p]), T_init=T[s], M=M[s], **kw)
        torch.testing.assert_close(got.plan[s], one.plan, rtol=1e-11, atol=1e-15)


def test_products_that_cancel():
    """Structures far from zero, whose products and constant part agree in all
    but their last digits.  Both are sums of integers here, exact in float64, so
    one step is a projection of exp(log T - lin / reg) with exponents up to 100:
    some tens of roundings of 2^7 2^-53 in K, u and v, 1e-12 relative in the plan."""
    rng = np.random.default_rng(7)
    n = m = 8
    C1 = 1000.0 + rng.integers(0, 5, (2, n, n))
    C2 = 1000.0 + rng.integers(0, 5, (2, m, m))
    C1, C2 = C1 + C1.transpose(0, 2, 1), C2 + C2.transpose(0, 2, 1)
    reg = 0.3
    T = np.full((2, n, m), 1.0 / (n * m))
    # sum_jl (C1_ij - C2_kl)^2 T_jl, formed without cancellation
    lin = 2.0 * np.einsum("bijkl->bik", (C1[:, :, :, None, None] - C2[:, None, None]) ** 2
                          ) / (n * m)
    K = np.log(T + 1e-15) - lin / reg
    v = np.zeros((2, m))
    for _ in range(30):
        u = np.log(1.0 / n) - np.logaddexp.reduce(K + v[:, None, :], axis=2)
        v = np.log(1.0 / m) - np.logaddexp.reduce(K + u[:, :, None], axis=1)
    want = np.exp(K + u[:, :, None] + v[:, None, :])
    got = pb.solve_gromov_batch(C1, C2, reg=reg, max_iter=1, max_iter_inner=30, tol_inner=0.0)
    np.testing.assert_allclose(got.plan, want, rtol=1e-12, atol=1e-18)
