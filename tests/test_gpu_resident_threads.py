"""Register-resident solves of several threads and streams at once.

The workgroups of a solve of several blocks wait for each other, so the solves
under way share the CUs; each gives the bits that it gives alone.
"""

import threading
import time

import pytest
import torch

from pot_amd import _lib, _solve

pytestmark = pytest.mark.gpu


def _problem(B, n, m, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    kw = dict(generator=g, device="cuda", dtype=torch.float64)
    M = torch.rand(B, n, m, **kw)
    a, b = torch.rand(B, n, **kw) + 0.2, torch.rand(B, m, **kw) + 0.2
    return M, a / a.sum(1, keepdim=True), b / b.sum(1, keepdim=True)


def _run(problem, iters):
    M, a, b = problem
    r = _solve.dense_solve(M, a, b, torch.zeros_like(a), torch.zeros_like(b), 0.05,
                           domain=_lib.LOG, order=_lib.COL_FIRST, max_iter=iters, stop_thr=0.0)
    return r.u.clone(), r.v.clone()


def _in_threads(work):
    """Runs the functions at the same time, each on a stream of its own; their results."""
    out, go = [None] * len(work), threading.Barrier(len(work))

    def body(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                go.wait()
                out[k] = work[k]()
                torch.cuda.current_stream().synchronize()
        except BaseException as e:  # noqa: B902
            out[k] = e

    threads = [threading.Thread(target=body, args=(k,)) for k in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for r in out:
        if isinstance(r, BaseException):
            raise r
    return out


def test_threads_give_the_bits_of_lone_solves():
    """Solves that fit the GPU together, one that fills it, and a batch with one stop."""
    shapes = [(1, 300, 260), (1, 900, 1000), (1, 2048, 2048), (40, 60, 50)]
    problems = [_problem(*s, seed=k) for k, s in enumerate(shapes)]
    want = [_run(p, 45) for p in problems]
    torch.cuda.synchronize()
    got = _in_threads([lambda p=p: [_run(p, 45) for _ in range(12)] for p in problems])
    for w, rs in zip(want, got):
        for r in rs:
            assert torch.equal(r[0], w[0]) and torch.equal(r[1], w[1])


def test_work_queued_before_a_solve_holds_up_no_other():
    """A thread whose stream is busy for 2.5 s before its solve; another's solve
    meanwhile gives the bits that it gives alone."""
    first, second = _problem(1, 300, 260, 1), _problem(1, 2048, 2048, 2)
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    start.record()
    torch.cuda._sleep(10_000_000)
    end.record()
    torch.cuda.synchronize()
    cycles = int(10_000_000 * 2500.0 / start.elapsed_time(end))
    want = [_run(first, 45), _run(second, 45)]

    def late():
        torch.cuda._sleep(cycles)
        return _run(first, 45)

    def soon():
        time.sleep(0.2)
        return _run(second, 45)

    got = _in_threads([late, soon])
    for w, r in zip(want, got):
        assert torch.equal(r[0], w[0]) and torch.equal(r[1], w[1])
