"""Weights that leave no plan or a meaningless one, in the register-resident
solves: outcomes are the row sweep's and the oracle's."""

import warnings

import numpy as np
import pytest
import torch

import oracle.stabilized as ostab
import pot_amd
from pot_amd import _lib, _solve

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("n,m", [(5, 4), (60, 50), (400, 360)])
@pytest.mark.parametrize("order", [_lib.COL_FIRST, _lib.ROW_FIRST])
def test_no_weight_in_any_column(n, m, order, dtype):
    g = torch.Generator("cuda").manual_seed(n)
    M = torch.rand(1, n, m, generator=g, device="cuda", dtype=dtype)
    a = torch.full((1, n), 1.0 / n, device="cuda", dtype=F64)
    b = torch.zeros((1, m), device="cuda", dtype=F64)
    assert _lib.load().potamd_dense_resident(_lib.F32 if dtype == F32 else _lib.F64, 1, n, m)
    kw = dict(domain=_lib.LOG, order=order, max_iter=20, stop_thr=1e-9)
    tile = (256, 4, 0, 1) if m > 128 else (64, 4, 0, 1) if dtype == F32 else (64, 2, 0, 1)
    want = _solve.dense_solve(M, a, b, torch.zeros_like(a), torch.zeros_like(b), 0.05, tile=tile,
                              **kw)
    got = _solve.dense_solve(M, a, b, torch.zeros_like(a), torch.zeros_like(b), 0.05, **kw)
    assert (got.status, got.niter, got.errs) == (want.status, want.niter, want.errs)
    for x, y in ((got.u, want.u), (got.v, want.v)):
        torch.testing.assert_close(x, y, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m", [(1, 5, 4), (3, 60, 50), (1, 400, 360), (2100, 20, 33)])
def test_negative_column_weight_is_refused(B, n, m, dtype):
    """Its logarithm is no number: the log domain raises, rows first too."""
    g = torch.Generator("cuda").manual_seed(n)
    M = torch.rand(B, n, m, generator=g, device="cuda", dtype=dtype)
    a = torch.full((B, n), 1.0 / n, device="cuda", dtype=F64)
    b = torch.full((B, m), 1.0 / m, device="cuda", dtype=F64)
    b[B // 2, 1] = -0.1
    for order in (_lib.COL_FIRST, _lib.ROW_FIRST):
        for iters in (1, 25):
            with pytest.raises(_lib.LibraryError):
                _solve.dense_solve(M, a, b, torch.zeros_like(a), torch.zeros_like(b), 0.05,
                                   domain=_lib.LOG, order=order, max_iter=iters, stop_thr=0.0)


def _both(a, b, M, reg, **kw):
    with warnings.catch_warnings(record=True) as W:
        warnings.simplefilter("always")
        P, lg = pot_amd.sinkhorn(*(torch.tensor(x, device="cuda") for x in (a, b, M)), reg,
                                 method="sinkhorn_stabilized", log=True, warn=False, **kw)
        got = [str(w.message) for w in W]
    with warnings.catch_warnings(record=True) as W, np.errstate(all="ignore"):
        warnings.simplefilter("always")
        Q, lo = ostab.sinkhorn_stabilized(a, b, M, reg, log=True, warn=False, **kw)
        want = [str(w.message) for w in W]
    assert got == want and lg["n_iter"] == lo["n_iter"]
    np.testing.assert_allclose(P.cpu().numpy(), Q, rtol=1e-10, atol=1e-18, equal_nan=True)
    return want


@pytest.mark.parametrize("n,m", [(6, 5), (60, 50), (400, 360)])
def test_stabilized_negative_weight_is_over_tau_too(n, m):
    """max |u| decides about absorption, whose logarithm then is no number."""
    rng = np.random.default_rng(n)
    a, b = rng.dirichlet(np.ones(n)), rng.dirichlet(np.ones(m))
    a[0] = -2.0
    M = rng.random((n, m))
    for iters in (1, 2, 7):
        _both(a, b, M, 0.2, numItermax=iters, tau=abs(a[0]))


@pytest.mark.parametrize("n,m", [(6, 5), (60, 50), (400, 360)])
@pytest.mark.parametrize("iters", [1, 3])
def test_stabilized_row_without_weight_or_kernel(n, m, iters):
    """0 / 0 in a row's scaling, in the last iteration as in an earlier one."""
    rng = np.random.default_rng(n)
    a, b = rng.dirichlet(np.ones(n)), rng.dirichlet(np.ones(m))
    M = rng.random((n, m))
    a[1], M[1] = 0.0, 1e3
    assert _both(a, b, M, 0.05, numItermax=iters) == ["Numerical errors at iteration 0"]


def _outcome(M, a, b, tile=None, **kw):
    n, m = M.shape[1:]
    scal = kw["domain"] == _lib.SCALING
    u0 = torch.full_like(a, 1.0 / n) if scal else torch.zeros_like(a)
    v0 = torch.full_like(b, 1.0 / m) if scal else torch.zeros_like(b)
    try:
        r = _solve.dense_solve(M, a, b, u0, v0, 0.05, tile=tile, order=_lib.COL_FIRST, **kw)
    except _lib.LibraryError as e:
        return str(e)
    return r.status, r.niter, r.bad_iter, len(r.errs)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m", [(1, 5, 4), (4, 60, 50), (1, 400, 360), (2100, 9, 7)])
def test_update_after_a_check_decides_first(B, n, m, dtype):
    """Iterations that check and end (converged, or the last) with a column that
    cannot be updated: masses below the trusted range, weights that are no number."""
    g = torch.Generator("cuda").manual_seed(n)
    M = torch.rand(B, n, m, generator=g, device="cuda", dtype=dtype)
    a = torch.full((B, n), 1.0 / n, device="cuda", dtype=F64)
    b = torch.full((B, m), 1.0 / m, device="cuda", dtype=F64)
    nan = a.clone()
    nan[B // 2, 0] = float("nan")
    tile = (256, 4, 0, 1) if m > 128 else (64, 4, 0, 1) if dtype == F32 else (64, 2, 0, 1)
    for domain in (_lib.LOG, _lib.SCALING):
        for iters, stop in ((1, 0.0), (32, 1e-7)):
            kw = dict(domain=domain, max_iter=iters, stop_thr=stop,
                      err_norm=int(domain == _lib.SCALING))
            for x, y in ((a * 1e-302, b * 1e-302), (nan, b), (a, b)):
                assert _outcome(M, x, y, **kw) == _outcome(M, x, y, tile=tile, **kw)
