"""Captured calls of the kernels that take one matrix per workgroup (those with
more than 64 KB of LDS set an attribute at each launch) and of the large batches
beside them: replays with eager work between them, against the eager result."""
from __future__ import annotations

import pytest
import torch

import helpers as H
import veig

pytestmark = pytest.mark.gpu


def replay(run, outs):
    run()
    torch.cuda.synchronize()
    eager = [o.clone() for o in outs]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run()
    for _ in range(3):
        for o in outs:
            o.fill_(-7)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(eager, outs))
        _ = (outs[0] * 2).sum().item()


def new(*counts):
    return [torch.empty(c, dtype=torch.float64, device="cuda") for c in counts]


@pytest.mark.parametrize("n,N", [(8, 6), (20, 300), (64, 6), (79, 6), (79, 516), (96, 6)])
def test_solve(gpu, n, N):
    rA, iA = (torch.from_numpy(x).cuda() for x in H.to_soa(H.gaussian(N, n, 950 + n), 2))
    outs = new(N * n, N * n, N * n * n, N * n * n)
    replay(lambda: veig.zgeev(rA, iA, n, N // 2, 2, out=tuple(outs)), outs)


@pytest.mark.parametrize("n,N", [(8, 6), (20, 300), (40, 6), (64, 6), (88, 6), (96, 6)])
def test_stages_and_values(gpu, n, N):
    rA, iA = (torch.from_numpy(x).cuda() for x in H.to_soa(H.gaussian(N, n, 970 + n), 2))
    outs = new(*[N * n * n] * 4, *[N * n] * (4 if n <= 64 else 2))

    def run():
        rH, iH, rZ, iZ, rE, iE = outs[:6]
        rH.copy_(rA)
        iH.copy_(iA)
        veig.hessenberg(n, N // 2, 2, rH, iH, rZ, iZ)
        veig.zlahqr(n, N // 2, 2, rE, iE, rH, iH, rZ, iZ)
        veig.ztrevc(n, N // 2, 2, rH, iH, rZ, iZ)
        if n <= 64:
            veig.eigvals(rA, iA, n, N // 2, 2, out=tuple(outs[6:]))

    replay(run, outs)
