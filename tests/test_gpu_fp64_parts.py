"""What is formed in fp64 for float32 costs too: the elements of the plan."""

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
