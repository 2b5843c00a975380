"""The streamed dense solve (csrc/dense.hip) on rows that do not end on a vector
of four (or two) elements or start on a 16-byte boundary, against the float64
oracle.

float64: the plan to 1e-11 relative (the sums are added in another order: a few
ulp an iteration).  float32: to 1e-5 relative on entries >= 1e-30, the bar of
the float32 solver.  Both domains are held to the log-domain oracle: their
iterations have the same plans, and only it takes zero weights on both sides.
"""

import numpy as np
import pytest
import torch

import oracle.sinkhorn as osk
from pot_amd import _lib, _solve, autotune

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
TILES = {F32: [(64, 4), (256, 4), (256, 8), (512, 8)], F64: [(64, 2), (256, 2), (256, 4), (512, 4)]}


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("n,m,pad", [(5, 1, 0), (5, 2, 0), (9, 3, 1), (7, 5, 0), (40, 255, 0),
                                     (33, 257, 2), (70, 1022, 3), (300, 1027, 0), (19, 1500, 1)])
def test_ragged_rows(n, m, pad, dtype):
    rng = np.random.default_rng(100 * n + m)
    B, reg = 2, 0.05
    wide = torch.tensor(rng.random((B, n, m + pad)), device="cuda", dtype=dtype)
    M = wide[:, :, pad:]  # rows of stride m + pad, from element pad on
    a, b = 0.2 + rng.random((B, n)), 0.2 + rng.random((B, m))
    if m > 3:
        b[:, 1::4] = 0.0
    a[:, 2::3] = 0.0
    a, b = a / a.sum(1, keepdims=True), b / b.sum(1, keepdims=True)
    at, bt = torch.tensor(a, device="cuda"), torch.tensor(b, device="cuda")
    tile = next(t for t in TILES[dtype] if t[0] * t[1] >= m)
    for rpb in (4, 16):
        for domain in (_lib.LOG, _lib.SCALING):
            u0, v0 = torch.zeros_like(at), torch.zeros_like(bt)
            if domain == _lib.SCALING:
                u0, v0 = torch.full_like(at, 1.0 / n), torch.full_like(bt, 1.0 / m)
            r = _solve.dense_solve(M, at, bt, u0, v0, reg, domain=domain, order=_lib.COL_FIRST,
                                   max_iter=12, stop_thr=0.0, tile=tile + (rpb, 1))
            for p in range(B):
                M64 = M[p].double().cpu().numpy()
                with np.errstate(divide="ignore", invalid="ignore"):
                    P, _ = osk.sinkhorn_log(a[p], b[p], M64, reg, numItermax=12, stopThr=0.0,
                                            log=True, warn=False)
                u, v = r.u[p].cpu().numpy(), r.v[p].cpu().numpy()
                with np.errstate(divide="ignore"):
                    u, v = (np.log(u), np.log(v)) if domain == _lib.SCALING else (u, v)
                got = np.exp(-M64 / reg + u[:, None] + v[None, :])
                mask = P >= 1e-30
                assert np.array_equal(got >= 1e-29, P >= 1e-29)
                rel = np.max(np.abs(got[mask] - P[mask]) / P[mask])
                assert rel < (1e-5 if dtype == F32 else 1e-11), (domain, p, rel)


def test_tile_keeps_its_workgroups(monkeypatch):
    """A cached tile serves the wide rows of its class with the number of
    workgroups that it was timed with; one without its sizes, as it is."""
    key = autotune._key("f32", 16384, 16384)
    monkeypatch.setattr(autotune, "_mem", {key: {"tile": [512, 32, 64, 1], "n": 16384, "m": 16384}})
    assert autotune.lookup("f32", 16384, 16384) == (512, 32, 64, 1)
    assert autotune.lookup("f32", 12000, 14336) == (512, 32, 47, 1)
    assert autotune.lookup("f32", 8193, 16000) == (512, 32, 33, 1)
    assert autotune.lookup("f32", 16384, 14335) is None
    monkeypatch.setattr(autotune, "_mem", {key: {"tile": [512, 32, 64, 1]}})
    assert autotune.lookup("f32", 12000, 9000) == (512, 32, 64, 1)
