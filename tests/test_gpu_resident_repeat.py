"""Register-resident solves that are given up and repeated: by a wait that ran
out, and by numbers that the row sweep has to report.  The repeat starts from the
caller's state, so it gives the row sweep's bits."""

import numpy as np
import pytest
import torch

import oracle.stabilized as ostab
import pot_amd
from pot_amd import _lib, _solve

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64


def _problem(B, n, m, dtype, seed):
    rng = np.random.default_rng(seed)
    M = torch.tensor(rng.random((B, n, m)), dtype=dtype, device="cuda")
    a, b = (torch.tensor(0.2 + rng.random((B, k)), device="cuda") for k in (n, m))
    return M, a / a.sum(1, keepdim=True), b / b.sum(1, keepdim=True)


def _run(M, a, b, domain, order, row_sweep=False, reg=0.05, **kw):
    m = M.shape[2]
    tiles = [(64, 4), (256, 4), (256, 8)] if M.dtype == F32 else [(64, 2), (256, 2), (256, 4)]
    tile = next(t for t in tiles if t[0] * t[1] >= m) + (0, 1) if row_sweep else None
    # (a start that is not the usual one)
    s = torch.linspace(0.5, 1.5, a.shape[1], dtype=F64, device="cuda")
    u0 = (torch.log(s) if domain == _lib.LOG else s / a.shape[1]).expand_as(a)
    v0 = torch.zeros_like(b) if domain == _lib.LOG else torch.full_like(b, 1.0 / m)
    return _solve.dense_solve(M, a, b, u0, v0, reg, domain=domain, order=order, tile=tile, **kw)


def _same(got, want):
    assert (got.status, got.niter, got.bad_iter) == (want.status, want.niter, want.bad_iter)
    assert got.errs == want.errs
    for x, y in ((got.u, want.u), (got.v, want.v)):  # (a column of zeros leaves a NaN in v)
        torch.testing.assert_close(x, y, rtol=0, atol=0, equal_nan=True)


@pytest.fixture
def giving_up():
    lib = _lib.load()
    lib.potamd_resident_wait_limit(-1)
    yield lib
    lib.potamd_resident_wait_limit(0)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m", [(1, 400, 360), (1, 30, 700), (1, 700, 30), (5, 400, 360),
                                   (40, 60, 50)])
@pytest.mark.parametrize("domain", [_lib.LOG, _lib.SCALING])
def test_a_wait_that_runs_out(B, n, m, dtype, domain, giving_up):
    problem = _problem(B, n, m, dtype, n)
    for order in (_lib.COL_FIRST, _lib.ROW_FIRST):
        kw = dict(domain=domain, order=order, max_iter=45, stop_thr=0.0)
        giving_up.potamd_resident_wait_limit(0)
        resident = _run(*problem, **kw)
        want = _run(*problem, row_sweep=True, **kw)
        assert not torch.equal(resident.u, want.u)  # (so the bits tell them apart)
        giving_up.potamd_resident_wait_limit(-1)
        _same(_run(*problem, **kw), want)
        # The device's solves do without waits for a while ...
        later = _run(*problem, **kw)
        if n * m > 128 * 128:  # (a batch of small ones runs in segments then)
            _same(later, want)
        # ... which ends with the call that sets the limit.
        giving_up.potamd_resident_wait_limit(0)
        _same(_run(*problem, **kw), resident)


@pytest.mark.parametrize("dtype", [F64, F32])
def test_a_wait_that_runs_out_stabilized(dtype, giving_up):
    """The repeat starts from the caller's alpha and beta."""
    M, a, b = _problem(1, 400, 360, dtype, 3)
    rng = np.random.default_rng(4)
    warm = 0.01 * rng.random(400), 0.01 * rng.random(360)
    P, log = ostab.sinkhorn_stabilized(a[0].cpu().numpy(), b[0].cpu().numpy(),
                                       M[0].double().cpu().numpy(), 0.01, numItermax=30, tau=3.0,
                                       warmstart=warm, log=True, warn=False)
    got, lg = pot_amd.sinkhorn(a[0], b[0], M[0], 0.01, method="sinkhorn_stabilized",
                               numItermax=30, tau=3.0, log=True, warn=False,
                               warmstart=tuple(torch.tensor(x, device="cuda") for x in warm))
    tol = 1e-10 if dtype == F64 else 1e-5
    assert np.max(np.abs(got.double().cpu().numpy() - P)) < tol * P.max()
    for key in ("alpha", "beta"):
        assert np.max(np.abs(lg[key].double().cpu().numpy() - log[key])) < tol


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m,order,err_norm", [(1, 400, 360, _lib.COL_FIRST, 1),
                                                  (3, 30, 700, _lib.COL_FIRST, 1),
                                                  (40, 60, 50, _lib.ROW_FIRST, 0),
                                                  (2100, 20, 33, _lib.ROW_FIRST, 0)])
def test_a_column_of_zeros(B, n, m, order, err_norm, dtype):
    """In one block of several, one problem of a batch, and a batch that is solved
    an interval at a time (whose state has been overwritten by then)."""
    M, a, b = _problem(B, n, m, dtype, B)
    M[B // 2, :, m - 2] = 1e6
    kw = dict(domain=_lib.SCALING, order=order, max_iter=50, stop_thr=0.0, err_norm=err_norm)
    want = _run(M, a, b, row_sweep=True, **kw)
    assert want.status == _lib.NUMERICAL
    _same(_run(M, a, b, **kw), want)
