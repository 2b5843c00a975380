"""The batched GEMM (csrc/batch_ops.hip) at the edges of its two tiles and K
chunks, against float64 products on the CPU.

A sum of K products rounded at every step is off by at most K eps of the sum of
the products' sizes; alpha and beta C add three roundings.
"""

import pytest
import torch

from pot_amd import _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 1, 1), (3, 32, 32, 64), (2, 33, 31, 65), (5, 16, 17, 3),
                                     (2, 100, 1, 130), (300, 64, 33, 32), (70, 65, 129, 37),
                                     (260, 3, 40, 95), (130, 128, 64, 1), (400, 20, 20, 20)])
def test_gemm(B, M, N, K, dtype):
    g = torch.Generator().manual_seed(1000 * M + N + K)
    eps = 2.0 ** (-53 if dtype == torch.float64 else -24)
    for tA in (False, True):
        for tB in (False, True):
            # every second column of a wider operand: no stride is 1
            wide = tA != tB
            A = torch.randn(B, *((K, M) if tA else (M, K)), 1 + wide, generator=g).to(dtype)[..., 0]
            Bm = torch.randn(B, *((N, K) if tB else (K, N)), 1 + wide, generator=g).to(dtype)[..., 0]
            C = torch.randn(B, M, N, generator=g).to(dtype)
            a = A.double().transpose(1, 2) if tA else A.double()
            b = Bm.double().transpose(1, 2) if tB else Bm.double()
            alpha, beta = 1.5, -0.25
            want = alpha * (a @ b) + beta * C.double()
            size = alpha * (a.abs() @ b.abs()) + abs(beta) * C.double().abs()
            # (device copies keep the strides of a sliced tensor only through its base)
            dev = [torch.empty_strided(t.shape, t.stride(), dtype=dtype, device="cuda") for t in (A, Bm)]
            for d, t in zip(dev, (A, Bm)):
                d.copy_(t)
            got = C.cuda()
            _solve.gemm(*dev, got, alpha=alpha, beta=beta, transA=tA, transB=tB)
            assert ((got.double().cpu() - want).abs() <= (K + 3) * eps * 1.01 * size).all()
            nan = torch.full_like(got, float("nan"))
            _solve.gemm(*dev, nan, transA=tA, transB=tB)
            one = a @ b
            assert ((nan.double().cpu() - one).abs() <= (K + 3) * eps * 1.01 * (a.abs() @ b.abs())).all()
