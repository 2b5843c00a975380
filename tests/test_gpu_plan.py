"""The plan kernel and its sums against numpy float64, at sizes where its
column threads, row blocks and vector loads end in the middle.

float64: 1e-12 relative (one exponential, sums of a few thousand terms);
float32 plans: half an ulp of the stored value, 6e-8, and the 2^-33 of the
exponential."""

import numpy as np
import pytest
import torch

from pot_amd import _lib, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,n,m", [(1, 1, 1), (3, 5, 7), (2, 70, 32), (600, 9, 16), (1, 37, 1026),
                                   (1, 3, 9000), (1, 300, 515)])
def test_plan_and_sums(B, n, m, dtype):
    rng = np.random.default_rng(n * m)
    M = rng.random((B, n, m)).astype(np.float32 if dtype == torch.float32 else np.float64)
    u, v = -5 + rng.standard_normal((B, n)), -4 + rng.standard_normal((B, m))
    u[0, 0] = -np.inf
    a, b = rng.random((B, n)) + 0.1, rng.random((B, m)) + 0.1
    reg = 0.07
    d = dict(device="cuda")
    Mt = torch.tensor(M, **d)
    ut, vt, at, bt = (torch.tensor(x, **d) for x in (u, v, a, b))
    tol = 1e-12 if dtype == torch.float64 else 7e-8
    for domain in (_lib.LOG, _lib.SCALING):
        for given in (False, True):
            Mk = Mt if not given else (-Mt / reg if domain == _lib.LOG else torch.exp(-Mt / reg))
            K = Mk.double().cpu().numpy()
            if domain == _lib.LOG:
                ux, vx = ut, vt
                x = (K if given else -K / reg) + u[:, :, None] + v[:, None, :]
                want = np.exp(x)
            else:
                ux, vx = torch.exp(ut), torch.exp(vt)
                want = np.exp(u)[:, :, None] * (K if given else np.exp(-K / reg)) \
                    * np.exp(v)[:, None, :]
            kw = dict(domain=domain, kernel_given=given, a=at, b=bt)
            alone, L, none = _solve.plan(Mk, ux, vx, reg, want_sums=0,
                                         want_log=domain == _lib.LOG, **kw)
            P, _, sums = _solve.plan(Mk, ux, vx, reg, **kw)
            assert none is None
            for got in (alone, P):
                np.testing.assert_allclose(got.double().cpu().numpy(), want, rtol=tol, atol=1e-44)
            if L is not None:
                np.testing.assert_allclose(L.double().cpu().numpy(), x, rtol=tol)
            with np.errstate(divide="ignore"):
                ref = np.stack([(K * want).sum((1, 2)), (want * np.log(want + 1e-16)).sum((1, 2)),
                                (want * np.log(want / (a[:, :, None] * b[:, None, :]) + 1e-16)
                                 ).sum((1, 2)), want.sum((1, 2))], 1)
            got = sums.cpu().numpy()
            scale = np.abs(ref).max()
            np.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-12 * scale)
            cost = _solve.plan(Mk, ux, vx, reg, want_plan=False, want_sums=_solve.SUM_COST,
                               **kw)[2].cpu().numpy()
            np.testing.assert_array_equal(cost[:, [0, 3]], got[:, [0, 3]])
            assert np.all(cost[:, 1:3] == 0)
