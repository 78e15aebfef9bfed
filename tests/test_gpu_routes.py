"""Both sides of the rules that send a batch to the lane-group kernels or to
one matrix per workgroup (few_matrices, per_workgroup): one matrix per CU (256)
for the entries with Schur vectors, four (1,024) without, and the stages above
order 16.  The same matrices alone (few) and repeated over a batch past the line
(many), against the oracle at the bar of test_gpu_parity and against each other."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
import veig
from gpu_util import gpu_eig
from test_gpu_parity import check_parity

pytestmark = pytest.mark.gpu
ORDERS = [7, 8, 9, 12, 13, 16, 17, 24, 25, 28, 29, 32]


def planes(A, tc):
    return tuple(torch.from_numpy(x).cuda() for x in H.to_soa(A, tc))


def values(rE, iE, n, tc):
    return H.vec_from_soa(rE.cpu().numpy(), iE.cpu().numpy(), n, tc)


@pytest.mark.parametrize("n", ORDERS)
def test_solve_past_one_matrix_per_cu(gpu, n):
    A = H.gaussian(13, n, 8000 + n)
    big = np.tile(A, (20, 1, 1))  # 260
    Eo, Vo, _ = H.oracle_eig(A, 1)
    for tc in (1, 13):
        E, V, info = gpu_eig(A, tc)
        check_parity(A, E, V, info, Eo, Vo)
        E, V, info = gpu_eig(big, tc)
        check_parity(A, E[:13], V[:13], info[:13], Eo, Vo)
        check_parity(A, E[-13:], V[-13:], info[-13:], Eo, Vo)
        assert np.all(info == 0)
        assert np.all(np.abs(E.reshape(20, 13, n) - E[:13]) <= 1e-12 * np.linalg.norm(A, axis=(1, 2))[:, None])


@pytest.mark.parametrize("n", ORDERS)
def test_schur_form_past_one_matrix_per_cu(gpu, n):
    A = H.gaussian(5, n, 8100 + n)
    big = np.tile(A, (52, 1, 1))
    for B in (A, big):
        E, V, info, T = gpu_eig(B, 1, write_schur=True)
        assert np.all(info == 0) and np.max(np.abs(np.tril(T, -1))) == 0.0
        assert np.allclose(np.diagonal(T, axis1=1, axis2=2), E, atol=0)


@pytest.mark.parametrize("n", [3, 4] + ORDERS)
def test_values_and_roots_past_four_matrices_per_cu(gpu, n):
    A = H.gaussian(5, n, 8200 + n)
    Eo, _, _ = H.oracle_eig(A, 5)
    norm = np.linalg.norm(A, axis=(1, 2))
    c = H.gaussian(5, n + 1, 8300 + n)[:, 0, :]
    first = None
    for rep in (1, 52, 206):  # 5, 260, 1,030
        B = np.tile(A, (rep, 1, 1))
        N = 5 * rep
        E = values(*veig.eigvals(*planes(B, 5), n, N // 5, 5), n, 5)
        _, err = H.match_eigenvalues(np.tile(Eo, (rep, 1)), E)
        assert np.all(err <= 1e-11 * np.tile(norm, rep))
        C = np.tile(c, (rep, 1))
        rC, iC = (torch.from_numpy(np.ascontiguousarray(x)).cuda().reshape(-1) for x in (C.real, C.imag))
        R = values(*veig.roots(rC, iC, n, N, 1), n, 1)
        first = R if first is None else first
        _, err = H.match_eigenvalues(np.tile(first, (rep, 1)), R)
        assert np.all(err <= 1e-9 * np.tile(np.abs(first).max(axis=1), rep))


@pytest.mark.parametrize("n", ORDERS)
@pytest.mark.parametrize("N", [6, 258, 1026])
def test_stages_either_side(gpu, n, N):
    A = np.tile(H.gaussian(6, n, 8400 + n), (N // 6, 1, 1))
    rH, iH = planes(A, 6)
    rZ, iZ = torch.empty_like(rH), torch.empty_like(iH)
    back = lambda r, i: H.from_soa(r.cpu().numpy(), i.cpu().numpy(), n, 6)  # noqa: E731
    herm = lambda X: np.conj(np.swapaxes(X, 1, 2))  # noqa: E731
    veig.hessenberg(n, N // 6, 6, rH, iH, rZ, iZ)
    Hs, Q = np.triu(back(rH, iH), -1), back(rZ, iZ)
    norm = np.linalg.norm(A, axis=(1, 2))
    tol = 1e-13 * n
    assert np.all(np.linalg.norm(Q @ herm(Q) - np.eye(n), axis=(1, 2)) <= tol)
    assert np.all(np.linalg.norm(A @ Q - Q @ Hs, axis=(1, 2)) <= tol * norm)
    rE, iE = (torch.empty(N * n, dtype=torch.float64, device="cuda") for _ in range(2))
    info = torch.full((N,), -1, dtype=torch.int32, device="cuda")
    veig.zlahqr(n, N // 6, 6, rE, iE, rH, iH, rZ, iZ, info=info)
    T, Z, E = np.triu(back(rH, iH)), back(rZ, iZ), values(rE, iE, n, 6)
    assert int((info != 0).sum()) == 0
    assert np.all(np.linalg.norm(Z @ herm(Z) - np.eye(n), axis=(1, 2)) <= tol)
    assert np.all(np.linalg.norm(A @ Z - Z @ T, axis=(1, 2)) <= tol * norm)
    veig.ztrevc(n, N // 6, 6, rH, iH, rZ, iZ)
    V = back(rZ, iZ)
    assert np.all(H.backward_error(A, E, V) <= 64 * n * np.finfo(float).eps)


@pytest.mark.parametrize("n", [65, 66, 79, 80])
def test_orders_above_64_past_two_matrices_per_cu(gpu, n):
    # few: four segments of 20 columns per Schur vector; many: two of 40
    A = H.gaussian(4, n, 8500 + n)
    big = np.tile(A, (129, 1, 1))  # 516
    Eo, Vo, _ = H.oracle_eig(A, 1)
    E, V, info = gpu_eig(big, 4)
    assert np.all(info == 0)
    check_parity(A, E[:4], V[:4], info[:4], Eo, Vo)
    check_parity(A, E[-4:], V[-4:], info[-4:], Eo, Vo)
    N = len(big)
    rH, iH = planes(big, 4)
    rZ, iZ = torch.empty_like(rH), torch.empty_like(iH)
    rE, iE = (torch.empty(N * n, dtype=torch.float64, device="cuda") for _ in range(2))
    veig.hessenberg(n, N // 4, 4, rH, iH, rZ, iZ)
    veig.zlahqr(n, N // 4, 4, rE, iE, rH, iH, rZ, iZ)
    Es = values(rE, iE, n, 4)
    veig.ztrevc(n, N // 4, 4, rH, iH, rZ, iZ)
    Vs = H.from_soa(rZ.cpu().numpy(), iZ.cpu().numpy(), n, 4)
    assert np.all(H.backward_error(big, Es, Vs) <= 64 * n * np.finfo(float).eps)
