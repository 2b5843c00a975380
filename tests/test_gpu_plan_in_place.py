"""A plan written over its own cost (P = M), as the C entry point takes it."""

import ctypes

import pytest
import torch

from pot_amd import _device, _lib, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,m", [(37, 1026), (3000, 2051), (64, 515), (64, 512)])
def test_plan_over_the_cost(n, m, dtype):
    """Rows that do not end with a 16-byte vector: an element is still read
    before it is written, and only then."""
    lib = _lib.load()
    g = torch.Generator("cuda").manual_seed(n)
    M = torch.rand(1, n, m, generator=g, device="cuda", dtype=dtype)
    u = torch.randn(1, n, generator=g, device="cuda", dtype=torch.float64)
    v = torch.randn(1, m, generator=g, device="cuda", dtype=torch.float64)
    want = _solve.plan(M, u, v, 0.5, domain=_lib.LOG, want_sums=0)[0]
    nbytes = lib.potamd_plan_workspace_size(1, n)
    ws = _device.workspace(nbytes, M.device)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    rc = lib.potamd_plan_dense(_lib.F32 if dtype == torch.float32 else _lib.F64, _lib.LOG, 0,
                               p(M), m, n * m, 1, n, m, 0.5, p(u), p(v), None, None, p(M), None,
                               n * m, None, p(ws), nbytes,
                               ctypes.c_void_p(_device.stream_ptr(M.device)))
    assert rc == 0
    assert torch.equal(M, want)
