"""What is formed in fp64 for float32 costs too: the elements of the plan, and
the first column update of the log domain."""

import numpy as np
import pytest
import torch

from pot_amd import _lib, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(70, 33), (300, 515), (2, 3)])
@pytest.mark.parametrize("domain", [_lib.LOG, _lib.SCALING])
def test_plan_is_the_same_with_and_without_sums(n, m, domain):
    g = torch.Generator("cuda").manual_seed(n)
    M = torch.rand(4, n, m, generator=g, device="cuda")
    u = torch.randn(4, n, generator=g, device="cuda", dtype=torch.float64) - 5
    v = torch.randn(4, m, generator=g, device="cuda", dtype=torch.float64) - 4
    if domain == _lib.SCALING:
        u, v = torch.exp(u), torch.exp(v)
    for reg in (0.003, 0.07):
        alone = _solve.plan(M, u, v, reg, domain=domain, want_sums=0)[0]
        both = _solve.plan(M, u, v, reg, domain=domain)[0]
        assert torch.equal(alone, both)


@pytest.mark.parametrize("n,m", [(40, 50), (300, 260), (30, 700)])
def test_first_column_update(n, m):
    """One iteration, columns first: v is one fp64 log-sum-exp of the given cost
    (exponents up to 1 / reg = 100, some roundings of 2^7 2^-53 and n of the
    sum's: 1e-12)."""
    rng = np.random.default_rng(n + m)
    M = rng.random((1, n, m)).astype(np.float32)
    a, b = rng.dirichlet(np.ones(n), 1), rng.dirichlet(np.ones(m), 1)
    d = dict(device="cuda")
    assert _lib.load().potamd_dense_resident(_lib.F32, 1, n, m)
    zero = torch.zeros
    r = _solve.dense_solve(torch.tensor(M, **d), torch.tensor(a, **d), torch.tensor(b, **d),
                           zero((1, n), dtype=torch.float64, **d),
                           zero((1, m), dtype=torch.float64, **d), 0.01, domain=_lib.LOG,
                           order=_lib.COL_FIRST, max_iter=1, stop_thr=0.0)
    want = np.log(b) - np.logaddexp.reduce(-M.astype(np.float64) / 0.01, axis=1)
    np.testing.assert_allclose(r.v.cpu().numpy(), want, atol=1e-12, rtol=0)
