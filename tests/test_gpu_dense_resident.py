"""The dense solve that keeps its cost in registers (csrc/dense_resident.hip)
at the edges of its tiles, against the float64 oracle, and its rarer ways
(references that move, exact row sums, segments of a batch too large to be
resident) against the row sweep on the same inputs.

float64: potentials to 1e-11 (the sums are added in another order: a few ulp
an iteration).  float32: the plan to 1e-5 relative on entries >= 1e-30, the
bar of the float32 solver.
"""

import numpy as np
import pytest
import torch

import oracle.batch as ob
import oracle.sinkhorn as osk
import oracle.stabilized as ostab
import pot_amd
from pot_amd import _lib, _solve

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
ROW_TILES = {F32: [(64, 4), (256, 4), (256, 8), (512, 8)],
             F64: [(64, 2), (256, 2), (256, 4), (512, 4)]}


def _problem(B, n, m, dtype, seed, zeros=False):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((B, n, 2))
    y = rng.standard_normal((B, m, 2)) + 1.0
    M = ((x[:, :, None] - y[:, None]) ** 2).sum(-1)
    M = (M / M.max((1, 2), keepdims=True)).astype(np.float32 if dtype == F32 else np.float64)
    a, b = 0.2 + rng.random((B, n)), 0.2 + rng.random((B, m))
    if zeros:
        a[:, ::3] = 0.0
        b[:, 1::4] = 0.0
    return M, a / a.sum(1, keepdims=True), b / b.sum(1, keepdims=True)


def _solve_gpu(M, a, b, reg, domain, order, row_sweep=False, **kw):
    d = dict(device="cuda")
    Mt, at, bt = torch.tensor(M, **d), torch.tensor(a, **d), torch.tensor(b, **d)
    B, n, m = Mt.shape
    code = _lib.F32 if Mt.dtype == F32 else _lib.F64
    assert _lib.load().potamd_dense_resident(code, B, n, m) == 1
    u0, v0 = torch.zeros_like(at), torch.zeros_like(bt)
    if domain == _lib.SCALING:
        u0, v0 = torch.full_like(at, 1.0 / n), torch.full_like(bt, 1.0 / m)
    tile = None
    if row_sweep:
        tile = next(t for t in ROW_TILES[Mt.dtype] if t[0] * t[1] >= m) + (0, 1)
    return _solve.dense_solve(Mt, at, bt, u0, v0, reg, domain=domain, order=order, tile=tile, **kw)


def _check_plan(M, reg, lu, lv, P, dtype):
    got = np.exp(-M.astype(np.float64) / reg + lu[:, None] + lv[None, :])
    mask = P >= 1e-30
    rel = np.max(np.abs(got[mask] - P[mask]) / P[mask])
    assert rel < (1e-5 if dtype == F32 else 1e-11), rel


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("n,m", [(1, 1), (16, 64), (33, 65), (64, 64), (65, 63), (128, 128),
                                 (129, 257), (256, 256), (257, 128), (20, 700), (900, 33)])
def test_single_problem(n, m, dtype):
    M, a, b = _problem(1, n, m, dtype, 1000 * n + m)
    M64 = M[0].astype(np.float64)
    reg = 0.05
    for domain in (_lib.LOG, _lib.SCALING):
        fn = osk.sinkhorn_log if domain == _lib.LOG else osk.sinkhorn_knopp
        P, log = fn(a[0], b[0], M64, reg, numItermax=25, stopThr=1e-4, log=True, warn=False)
        r = _solve_gpu(M, a, b, reg, domain, _lib.COL_FIRST, max_iter=25, stop_thr=1e-4,
                       err_norm=domain)
        assert r.niter == log["niter"] and len(r.errs) == len(log["err"])
        u, v = r.u[0].cpu().numpy(), r.v[0].cpu().numpy()
        if domain == _lib.SCALING:
            u, v = np.log(u), np.log(v)
        _check_plan(M[0], reg, u, v, P, dtype)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m", [(7, 48, 40), (300, 30, 64), (2100, 20, 33), (3, 300, 140)])
def test_batch_with_one_stop(B, n, m, dtype):
    """One launch, one launch per check interval (more problems than fit) and
    blocked problems: all stop together."""
    M, a, b = _problem(B, n, m, dtype, B)
    ref = ob.bregman_log_projection_batch(-M.astype(np.float64) / 0.05, a, b, max_iter=200,
                                          tol=1e-4)
    r = _solve_gpu(M, a, b, 0.05, _lib.LOG, _lib.ROW_FIRST, max_iter=200, stop_thr=1e-4)
    assert r.niter == ref["n_iters"]
    u, v = r.u.cpu().numpy(), r.v.cpu().numpy()
    for p in range(0, B, max(1, B // 5)):
        _check_plan(M[p], 0.05, u[p], v[p], ref["T"][p], dtype)
    ref = ob.bregman_projection_batch(np.exp(-M.astype(np.float64) / 0.1), a, b, max_iter=13,
                                      tol=0.0)
    r = _solve_gpu(M, a, b, 0.1, _lib.SCALING, _lib.ROW_FIRST, max_iter=13, stop_thr=0.0)
    assert r.niter == 12 and r.status == _lib.MAX_ITER
    f, g = r.u.cpu().numpy(), r.v.cpu().numpy()
    for p in range(0, B, max(1, B // 5)):
        _check_plan(M[p], 0.1, np.log(f[p]), np.log(g[p]), ref["T"][p], dtype)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("n,m,reg,zeros", [(120, 100, 0.002, False), (600, 500, 0.002, False),
                                           (120, 100, 0.02, True), (600, 500, 0.02, True),
                                           (200, 180, 0.0005, False)])
def test_references_and_exact_rows(n, m, reg, zeros, dtype):
    """Small reg: scalings leave their range and row sums the type's; zero
    weights give the same infinite potentials, and a column mass below the
    float32 range is refused by both."""
    M, a, b = _problem(1, n, m, dtype, n, zeros)
    for order in (_lib.COL_FIRST, _lib.ROW_FIRST):
        kw = dict(domain=_lib.LOG, order=order, max_iter=40, stop_thr=0.0)
        try:
            want = _solve_gpu(M, a, b, reg, row_sweep=True, **kw)
        except _lib.LibraryError:
            with pytest.raises(_lib.LibraryError):
                _solve_gpu(M, a, b, reg, **kw)
            continue
        got = _solve_gpu(M, a, b, reg, **kw)
        assert got.niter == want.niter and got.status == want.status
        for x, y in ((got.u, want.u), (got.v, want.v)):
            assert torch.equal(torch.isfinite(x), torch.isfinite(y))
            fin = torch.isfinite(y)
            # potentials up to 1/reg in size; float32 exponents carry their
            # rounding: 2^-24 of that each
            tol = 1e-11 / reg if dtype == F64 else 3e-7 / reg
            assert (x[fin] - y[fin]).abs().max().item() < max(tol, 2e-5 if dtype == F32 else 0.0)


@pytest.mark.parametrize("n,m,dtype", [(4801, 4500, F32), (5120, 5119, F32), (2816, 2900, F64)])
def test_largest_blocks(n, m, dtype):
    """Every CU holds a block; against the row sweep."""
    g = torch.Generator(device="cuda").manual_seed(n)
    M = torch.rand((1, n, m), generator=g, device="cuda", dtype=dtype)
    a = torch.rand((1, n), generator=g, device="cuda", dtype=torch.float64) + 0.2
    b = torch.rand((1, m), generator=g, device="cuda", dtype=torch.float64) + 0.2
    a, b = a / a.sum(), b / b.sum()
    assert _lib.load().potamd_dense_resident(_lib.F32 if dtype == F32 else _lib.F64, 1, n, m)
    tile = (1024, 8, 0, 1) if dtype == F32 else (1024, 4, 0, 1)
    for domain in (_lib.LOG, _lib.SCALING):
        u0, v0 = torch.zeros_like(a), torch.zeros_like(b)
        if domain == _lib.SCALING:
            u0, v0 = torch.full_like(a, 1.0 / n), torch.full_like(b, 1.0 / m)
        kw = dict(domain=domain, order=_lib.COL_FIRST, max_iter=12, stop_thr=0.0)
        want = _solve.dense_solve(M, a, b, u0, v0, 0.05, tile=tile, **kw)
        got = _solve.dense_solve(M, a, b, u0, v0, 0.05, **kw)
        for x, y in ((got.u, want.u), (got.v, want.v)):
            if domain == _lib.SCALING:
                x, y = torch.log(x), torch.log(y)
            # 12 iterations of sums of 5000 terms
            assert (x - y).abs().max().item() < (1e-11 if dtype == F64 else 5e-6)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m", [(2100, 30, 40), (5, 300, 260)])
def test_each_problem_stops_itself(B, n, m, dtype):
    M, a, b = _problem(B, n, m, dtype, B + 1)
    kw = dict(domain=_lib.LOG, order=_lib.COL_FIRST, max_iter=100, stop_thr=1e-3, each=True)
    want = _solve_gpu(M, a, b, 0.05, row_sweep=True, **kw)
    got = _solve_gpu(M, a, b, 0.05, **kw)
    same = got.niters == want.niters
    assert torch.equal(got.statuses[same], want.statuses[same])
    # float32 sums may cross the threshold one check apart
    assert (~same).sum().item() <= (0 if dtype == F64 else B // 100 + 1)
    assert (got.u - want.u)[same].abs().max().item() < (1e-10 if dtype == F64 else 2e-5)


def test_numerical_errors_are_the_row_sweeps():
    """A column of zeros in K: the solve is abandoned and the row sweep
    reports the reverted pair and the iteration."""
    M, a, b = _problem(1, 50, 60, F64, 5)
    M[0, :, 7] = 1e6
    kw = dict(domain=_lib.SCALING, order=_lib.COL_FIRST, max_iter=50, stop_thr=0.0, err_norm=1)
    want = _solve_gpu(M, a, b, 0.05, row_sweep=True, **kw)
    got = _solve_gpu(M, a, b, 0.05, **kw)
    assert got.status == want.status == _lib.NUMERICAL
    assert got.bad_iter == want.bad_iter and torch.equal(got.u, want.u)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("n,m,tau,iters", [(64, 64, 1e3, 1), (65, 33, 2.0, 45), (120, 100, 1e3, 80),
                                           (300, 260, 3.0, 60), (30, 700, 1e3, 41),
                                           (700, 30, 5.0, 41)])
def test_stabilized_absorbs_as_the_oracle(n, m, tau, iters, dtype):
    """Absorption now and then, at every iteration and in the last one, with
    one block and with rows or columns (or both) in several."""
    M, a, b = _problem(1, n, m, dtype, n + m)
    reg = 0.005
    P, log = ostab.sinkhorn_stabilized(a[0], b[0], M[0].astype(np.float64), reg, numItermax=iters,
                                       tau=tau, log=True, warn=False)
    got, lg = pot_amd.sinkhorn(torch.tensor(a[0], device="cuda"), torch.tensor(b[0], device="cuda"),
                               torch.tensor(M[0], device="cuda"), reg,
                               method="sinkhorn_stabilized", numItermax=iters, tau=tau, log=True,
                               warn=False)
    assert lg["n_iter"] == log["n_iter"] and len(lg["err"]) == len(log["err"])
    # float64: a few ulp of exponents up to 1 / reg an iteration; float32: K is
    # stored in float32
    tol = 1e-10 if dtype == F64 else 1e-5
    assert np.max(np.abs(got.cpu().numpy() - P)) < tol * P.max()
    for key in ("alpha", "beta"):
        assert np.max(np.abs(lg[key].double().cpu().numpy() - log[key])) < tol
    np.testing.assert_allclose([float(e) for e in lg["err"]], log["err"], rtol=max(tol, 1e-6),
                               atol=1e-12 if dtype == F64 else 1e-7)


@pytest.mark.parametrize("n,m,dtype", [(9000, 128, F64), (250, 8190, F64), (9000, 250, F32),
                                       (2801, 2790, F64)])
def test_many_values_to_exchange(n, m, dtype):
    """Column or row groups of so many values that their members add a part
    each and exchange the totals."""
    M, a, b = _problem(1, n, m, dtype, n + m)
    reg = 0.05
    for domain in (_lib.LOG, _lib.SCALING):
        fn = osk.sinkhorn_log if domain == _lib.LOG else osk.sinkhorn_knopp
        P, log = fn(a[0], b[0], M[0].astype(np.float64), reg, numItermax=12, stopThr=0.0, log=True,
                    warn=False)
        r = _solve_gpu(M, a, b, reg, domain, _lib.COL_FIRST, max_iter=12, stop_thr=0.0,
                       err_norm=domain)
        np.testing.assert_allclose(r.errs, log["err"], rtol=1e-9 if dtype == F64 else 1e-2,
                                   atol=1e-9 if dtype == F64 else 1e-6)
        u, v = r.u[0].cpu().numpy(), r.v[0].cpu().numpy()
        if domain == _lib.SCALING:
            u, v = np.log(u), np.log(v)
        _check_plan(M[0], reg, u, v, P, dtype)


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("B,n,m", [(300, 128, 127), (257, 65, 66)])
def test_more_problems_than_cus(B, n, m, dtype):
    """Problems of 65 to 128 a side, two and more of them on a CU."""
    test_batch_with_one_stop(B, n, m, dtype)
