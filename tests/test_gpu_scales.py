"""Matrices whose squares overflow or underflow, through the kernels that take
one matrix per workgroup: a power of two is exact, so E, T and H are those of
the matrix near 1 times it, V, Q and Z the same, to the bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
import veig
from gpu_util import gpu_eig

pytestmark = pytest.mark.gpu
EXPONENTS = [-960, -520, -480, 500, 900]


def planes(A):
    return tuple(torch.from_numpy(x).cuda() for x in H.to_soa(A, 1))


def zeros(count):
    return tuple(torch.zeros(count, dtype=torch.float64, device="cuda") for _ in range(2))


def back(p, n):
    return H.from_soa(p[0].cpu().numpy(), p[1].cpu().numpy(), n, 1)


def vec(p, n):
    return H.vec_from_soa(p[0].cpu().numpy(), p[1].cpu().numpy(), n, 1)


def same(a, b, s=1.0):
    # component by component: a product of complex numbers would round subnormals twice
    return np.array_equal(a.real * s, b.real) and np.array_equal(a.imag * s, b.imag) and bool(np.all(np.isfinite(b)))


@pytest.mark.parametrize("k", EXPONENTS)
@pytest.mark.parametrize("n", [8, 16, 17, 24, 32, 33, 48, 64, 65, 80, 96])
def test_solve(gpu, n, k):
    A = H.gaussian(2, n, 9800 + n)
    E, V, info, T = gpu_eig(A, 1, write_schur=True)
    Es, Vs, infos, Ts = gpu_eig(A * 2.0 ** k, 1, write_schur=True)
    assert np.all(info == 0) and np.all(infos == 0)
    assert same(E, Es, 2.0 ** k) and same(V, Vs) and same(T, Ts, 2.0 ** k)


@pytest.mark.parametrize("k", EXPONENTS)
@pytest.mark.parametrize("n,N", [(8, 2), (16, 2), (17, 2), (24, 1030), (32, 1030), (33, 2), (48, 2), (64, 2), (80, 2), (96, 2)])
def test_stages_and_values(gpu, n, N, k):
    A = np.tile(H.gaussian(2, n, 9900 + n), (N // 2, 1, 1))
    s = 2.0 ** k
    few = N == 2
    out = []
    for X in (A, A * s):
        a, q, e = planes(X), zeros(X.size), zeros(N * n)
        veig.hessenberg(n, N, 1, *a, *q)
        r = [np.triu(back(a, n), -1), back(q, n)]
        if few:
            z = tuple(x.clone() for x in q)
            veig.zlahqr(n, N, 1, *e, *a, *z)
            r += [vec(e, n), np.triu(back(a, n)), back(z, n)]
            if n > 16:  # (below: lane groups)
                veig.ztrevc(n, N, 1, *a, *z)
            r += [back(z, n)]
            if n <= 64:
                r += [vec(veig.eigvals(*planes(X), n, N, 1), n)]
                h = planes(r[0])
                r += [vec(veig.zlahqr_eig(*h, n, N, 1), n), np.triu(back(h, n), -1)]
        out.append(r)
    scaled = [True, False, True, True, False, False, True, True, True]
    for x, y, f in zip(*out, scaled):
        assert same(x, y, s if f else 1.0)


@pytest.mark.parametrize("n", [16, 33, 64, 80])
def test_subdiagonal_far_below_the_rest(gpu, n):
    # the reduction meets a column whose square underflows: nothing to reduce
    A = np.triu(H.gaussian(1, n, 9950 + n), -1)
    A[0, n // 2, n // 2 - 1] = 1e-200j
    E, V, info = gpu_eig(A, 1)
    assert np.all(info == 0) and np.all(np.isfinite(V))
    assert np.all(H.backward_error(A, E, V) <= 64 * n * np.finfo(float).eps)


@pytest.mark.parametrize("k", [-960, -700])
@pytest.mark.parametrize("route", ["batch", "uneven", "mixed"])
@pytest.mark.parametrize("n", [12, 16, 20, 24, 27, 28, 32])
def test_lane_groups_report_what_they_lose(gpu, n, route, k):
    # the QR iteration on lane groups does not scale: such a matrix is reported
    # (info) or undefined, never returned as converged and wrong
    A = np.tile(H.gaussian(3, n, 9970 + n) * 2.0 ** k, (101, 1, 1))
    if route == "uneven":
        from test_gpu_varsize import fetch
        vb = veig.VarBatch([n] * len(A))
        vb.rA.copy_(torch.from_numpy(np.ascontiguousarray(np.swapaxes(A, 1, 2)).reshape(-1).real.copy()))
        vb.iA.copy_(torch.from_numpy(np.ascontiguousarray(np.swapaxes(A, 1, 2)).reshape(-1).imag.copy()))
        vb.run()
        torch.cuda.synchronize()
        out = fetch(vb, [n] * len(A))
        E, V, info = np.stack([o[0] for o in out]), np.stack([o[1] for o in out]), vb.info.cpu().numpy()
    else:
        E, V, info = gpu_eig(A, 1, precision="mixed" if route == "mixed" else "fp64")[:3]
    silent = (info == 0) & np.all(np.isfinite(E), axis=1)
    if np.any(silent):
        want, _, _ = H.oracle_eig(A[silent] * 2.0 ** -k, 1)
        _, err = H.match_eigenvalues(want, E[silent] * 2.0 ** -k)
        assert np.all(err <= 1e-9 * np.linalg.norm(A[silent] * 2.0 ** -k, axis=(1, 2)))
