"""The kernels of large batches at orders 8..32 (k_zgeev<8>, k_gehrd_c or k_reduce,
then k_qr_band in slots of 12, 16, 24, 28 and 32: four or two matrices share a
wavefront) on the inputs that the other GPU tests give in batches of at most 256,
which take one matrix per workgroup: ragged counts, special matrices beside
ordinary ones in one wavefront, the Schur form, the iteration cap, long lists.
And, of the one-matrix-per-workgroup kernels, what no other test reaches: the
exceptional shifts in two slots of lanes and in segments of 40 and 48 columns,
and a complex subdiagonal made real."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
import veig
from gpu_util import gpu_eig
from test_gpu_mixed import run_mixed
from test_gpu_parity import check_parity, constructed, hermitian, unit_upper_eigvecs
from test_gpu_shifts import cyclic

pytestmark = pytest.mark.gpu
ORDERS = [8, 9, 12, 13, 16, 17, 24, 25, 28, 29, 32]  # edges of the slots
EPS = np.finfo(float).eps


def fill(A, N):
    """A repeated to N matrices (the last round cut)"""
    return np.concatenate([A] * (N // len(A) + 1))[:N]


@pytest.mark.parametrize("n", ORDERS)
@pytest.mark.parametrize("N", [257, 258, 259])
def test_ragged_counts(gpu, n, N):
    A = H.gaussian(11, n, 9000 + n)
    Eo, Vo, _ = H.oracle_eig(A, 1)
    E, V, info = gpu_eig(fill(A, N), 1)
    check_parity(fill(A, N), E, V, info, fill(Eo, N), fill(Vo, N))


@pytest.mark.parametrize("n", ORDERS)
@pytest.mark.parametrize("N", [263, 264])
def test_special_matrices_beside_ordinary_ones(gpu, n, N):
    G = H.gaussian(3, n, 9100 + n)
    tri = np.triu(H.gaussian(1, n, 9200 + n)[0]) + np.diag(3.0 * np.arange(n))
    hess = np.triu(H.gaussian(1, n, 9300 + n)[0], -1)
    hess[3, 2] = hess[n - 1, n - 2] = 0
    nan = H.gaussian(1, n, 9400 + n)[0]
    nan[n // 2, 1] = np.nan
    # seven to a round: every slot of a wavefront meets each
    base = np.stack([G[0], np.zeros((n, n), complex), tri, nan, G[1], hess, np.diag(np.arange(1, n + 1) + 0j)])
    A = fill(base, N)
    E, V, info = gpu_eig(A, 1)
    Eo, Vo, _ = H.oracle_eig(G, 1)
    kind = np.arange(N) % 7
    for k, g in ((0, 0), (4, 1)):
        m = kind == k
        c = int(m.sum())
        check_parity(A[m], E[m], V[m], info[m], np.repeat(Eo[g:g + 1], c, 0), np.repeat(Vo[g:g + 1], c, 0))
    assert np.all(E[kind == 1] == 0) and np.all(info[kind == 1] == 0)
    assert np.all((info[kind == 3] > 0) | ~np.all(np.isfinite(E[kind == 3]), axis=1))
    for k, want in ((2, np.diag(tri)), (5, np.linalg.eigvals(hess)), (6, np.arange(1, n + 1) + 0j)):
        m = kind == k
        assert np.all(info[m] == 0) and np.all(np.isfinite(V[m]))
        _, err = H.match_eigenvalues(np.repeat(want[None], int(m.sum()), 0), E[m])
        assert np.all(err <= 1e-9 * np.linalg.norm(base[k]))
        assert np.max(H.backward_error(A[m], E[m], V[m])) < 64 * n * EPS


@pytest.mark.parametrize("n", ORDERS)
def test_hermitian_constructed_clustered(gpu, n):
    for A, vec in ((hermitian(7, n, 9500 + n), False), (constructed(7, n, 9600 + n, cond=1e2), True),
                   (constructed(7, n, 9700 + n, cond=1e2, cluster=1e-6), False)):
        Eo, Vo, _ = H.oracle_eig(A, 1)
        E, V, info = gpu_eig(fill(A, 261), 1)
        check_parity(fill(A, 261), E, V, info, fill(Eo, 261), fill(Vo, 261), vec_check=vec)


@pytest.mark.parametrize("n", [n for n in ORDERS if n > 8])
def test_exceptional_shifts(gpu, n):
    A = H.gaussian(5, n, 9800 + n)
    A[1], A[3] = cyclic(n), cyclic(n, 2.0)
    Eo, Vo, _, (info_o, sweeps, _) = H.oracle_eig(A, 1, H.LAPACK_SIGN | H.LAPACK_TST, stats=True)
    assert np.all(info_o == 0)
    E, V, info = gpu_eig(fill(A, 263), 1)
    check_parity(fill(A, 263), E, V, info, fill(Eo, 263), fill(Vo, 263))


@pytest.mark.parametrize("n", ORDERS)
def test_schur_form(gpu, n):
    A = H.gaussian(3, n, 9900 + n)
    E, V, info, T = gpu_eig(fill(A, 259), 1, write_schur=True)
    assert np.all(info == 0) and np.all(np.tril(T, -1) == 0)
    assert np.array_equal(np.diagonal(T, 0, 1, 2), E)
    for m in (slice(0, 3), slice(256, 259)):
        B = fill(A, 259)[m]
        Z = V[m] @ np.linalg.inv(unit_upper_eigvecs(T[m]))
        assert np.max(np.linalg.norm(np.conj(np.swapaxes(Z, 1, 2)) @ Z - np.eye(n), axis=(1, 2))) < 1e-12 * n
        assert np.max(np.linalg.norm(B @ Z - Z @ T[m], axis=(1, 2)) / np.linalg.norm(B, axis=(1, 2))) < 1e-13 * n


@pytest.mark.parametrize("n", ORDERS)
def test_iteration_cap(gpu, n):
    A = H.gaussian(257, n, 10000 + n)
    _, _, info = gpu_eig(A, 1, itmax=1)
    assert np.any(info > 0)
    E, V, info = gpu_eig(A, 1)
    assert np.all(info == 0) and np.max(H.backward_error(A, E, V)) < 64 * n * EPS


@pytest.mark.parametrize("n", [12, 16, 20, 24, 27, 32, 40, 64])
def test_long_lists(gpu, n):
    # every third matrix of the batch goes to the FP64 solve of the list
    N = 601 if n <= 32 else 200
    A = H.gaussian(N, n, 10100 + n)
    A[::3] = fill(constructed(8, n, 10200 + n, cond=1e9), N)[::3]
    E, V, info, fb, be = run_mixed(A)
    assert np.all(info == 0) and fb[::3].mean() > 0.9 and fb.mean() < 0.7
    assert np.all(be <= 1e-12) and np.all(H.backward_error(A, E, V) <= 1e-12)


@pytest.mark.parametrize("n,N", [(34, 4), (66, 4), (79, 516), (88, 4), (96, 4)])
def test_exceptional_shifts_above_32(gpu, n, N):
    A = H.gaussian(4, n, 10300 + n)
    A[1], A[2] = cyclic(n), cyclic(n, 2.0)
    Eo, Vo, _, (info_o, sweeps, _) = H.oracle_eig(A, 1, H.LAPACK_SIGN | H.LAPACK_TST, stats=True)
    assert np.all(info_o == 0)
    assert sweeps[1] >= 11 + 2 * (n - 2), "the cyclic matrix must need the exceptional shift"
    E, V, info = gpu_eig(fill(A, N), 1)
    assert np.all(info == 0)
    for m in (slice(0, 4), slice(N - 4, N)):
        check_parity(A, E[m], V[m], info[m], Eo, Vo)


@pytest.mark.parametrize("n,N", [(n, N) for n in (8, 16, 24, 32) for N in (3, 259)] +
                         [(33, 3), (48, 3), (64, 3), (65, 3), (80, 3), (81, 3), (96, 3)])
def test_complex_subdiagonal(gpu, n, N):
    A = np.triu(H.gaussian(3, n, 10400 + n), -1)
    A[1, n // 2, n // 2 - 1] = 0
    A[2, 1:, :-1][np.arange(n - 1), np.arange(n - 1)] *= 1j ** np.arange(n - 1)
    B = fill(A, N)
    dev = lambda X: tuple(torch.from_numpy(x).cuda() for x in H.to_soa(X, 1))  # noqa: E731
    h, z = dev(B), dev(np.repeat(np.eye(n)[None] + 0j, N, 0))
    e = tuple(torch.empty(N * n, dtype=torch.float64, device="cuda") for _ in range(2))
    info = torch.full((N,), -1, dtype=torch.int32, device="cuda")
    veig.zlahqr(n, N, 1, *e, *h, *z, info=info)
    T, Z = (H.from_soa(p[0].cpu().numpy(), p[1].cpu().numpy(), n, 1) for p in (h, z))
    E = H.vec_from_soa(e[0].cpu().numpy(), e[1].cpu().numpy(), n, 1)
    norm = np.linalg.norm(B, axis=(1, 2))
    assert int((info != 0).sum()) == 0
    assert np.all(np.tril(T, -1) == 0) and np.array_equal(np.diagonal(T, 0, 1, 2), E)
    assert np.all(np.linalg.norm(np.conj(np.swapaxes(Z, 1, 2)) @ Z - np.eye(n), axis=(1, 2)) <= 1e-13 * n)
    assert np.all(np.linalg.norm(B @ Z - Z @ T, axis=(1, 2)) <= 1e-13 * n * norm)
