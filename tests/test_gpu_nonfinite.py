"""Infinities and NaN where an operation does not read them: what the reduction
has finished, what an eigenvector or a deflated block does not depend on.  The
rest of the result is finite and holds the properties that it has without them
(tolerances as in test_gpu_routes)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
import veig

pytestmark = pytest.mark.gpu
BAD = [np.inf, np.nan]


def planes(A):
    return tuple(torch.from_numpy(x).cuda() for x in H.to_soa(A, 1))


def zeros(count):
    return tuple(torch.zeros(count, dtype=torch.float64, device="cuda") for _ in range(2))


def back(p, n):
    return H.from_soa(p[0].cpu().numpy(), p[1].cpu().numpy(), n, 1)


def vec(p, n):
    return H.vec_from_soa(p[0].cpu().numpy(), p[1].cpu().numpy(), n, 1)


def norm(X):
    return np.linalg.norm(X, axis=(-2, -1))


# (order, matrices): one matrix per workgroup in every capacity, and the lane
# groups of the orders up to 16
SIZES = [(8, 3), (16, 3), (17, 3), (24, 3), (32, 3), (33, 3), (48, 3), (64, 3), (80, 3), (96, 3), (16, 1027)]


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("n,N", SIZES)
def test_reduction_first_row(gpu, n, N, bad):
    # no reflector and no update from the left reads row 0, and no update from
    # the right mixes it with others: Q and the rows below are those of the
    # matrix with any other first row
    A = np.tile(H.gaussian(1, n, 9000 + n), (N, 1, 1))
    for m, c in enumerate((0, n // 2, n - 1)):
        A[m, 0, c] = bad
    a, q = planes(A), zeros(A.size)
    veig.hessenberg(n, N, 1, *a, *q)
    b, t = planes(A), zeros(N * n)
    veig.zgehrd(n, N, 1, *b, *t)
    Hs, Q, tol = np.triu(back(a, n), -1), back(q, n), 1e-13 * n
    assert np.all(norm(Q @ np.conj(np.swapaxes(Q, 1, 2)) - np.eye(n)) <= tol)
    assert np.all(Q[:, 0, 1:] == 0) and np.all(Q[:, 1:, 0] == 0)
    R = A[:, 1:] @ Q - Q[:, 1:, 1:] @ Hs[:, 1:]
    assert np.all(norm(R) <= tol * norm(A[:, 1:]))
    assert np.array_equal(back(b, n)[:, 1:], back(a, n)[:, 1:])
    assert np.all(np.isfinite(vec(t, n)))


@pytest.mark.parametrize("n", [17, 24, 32, 33, 48, 64, 80, 96])
def test_q_columns_before_a_reflector(gpu, n):
    # reflector i changes columns i+1..n-1 of Q only
    a, t = planes(H.gaussian(1, n, 9100 + n)), zeros(n)
    veig.zgehrd(n, 1, 1, *a, *t)
    C = back(a, n)
    ref = planes(C)
    veig.zunghr(n, 1, 1, *ref, *t)
    for i in (0, 1, n // 2, n - 3):
        B = C.copy()
        B[0, n - 1, i] = np.nan
        q = planes(B)
        veig.zunghr(n, 1, 1, *q, *t)
        assert np.all(np.abs(back(ref, n) - back(q, n))[:, :, :i + 1] <= 1e-13 * n)


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("n", [16, 17, 24, 31, 32, 33, 48, 64, 65, 80, 96])
def test_eigenvectors_that_do_not_depend_on_it(gpu, n, bad):
    # eigenvector k depends on T(i, j) for i <= j <= k, row r of its result on R(r, j) for j <= k
    T = np.triu(H.gaussian(1, n, 9200 + n))[0] + np.diag(3.0 * np.arange(n))
    R = np.linalg.qr(H.gaussian(1, n, 9300 + n)[0])[0]
    ref = planes(R[None])
    veig.ztrevc(n, 1, 1, *planes(T[None]), *ref)
    ref, tol = back(ref, n)[0], 1e-13 * n
    for i, j in ((0, n // 2), (n // 2 - 1, n - 1), (n // 2, n // 2), (0, 1)):
        B = T.copy()
        B[i, j] = bad
        v = planes(R[None])
        veig.ztrevc(n, 1, 1, *planes(B[None]), *v)
        assert np.all(np.abs(back(v, n)[0] - ref)[:, :j] <= tol * np.abs(ref).max())
    for r, j in ((0, n - 1), (n - 1, n // 2), (n // 2, 1)):
        Z = R.copy()
        Z[r, j] = bad
        v = planes(Z[None])
        veig.ztrevc(n, 1, 1, *planes(T[None]), *v)
        diff = np.abs(back(v, n)[0] - ref)
        assert np.all(diff[r, :j] <= tol * np.abs(ref).max())
        assert np.all(np.delete(diff, r, axis=0) <= tol * np.abs(ref).max())


@pytest.mark.parametrize("n", [33, 48, 64, 65, 80, 96])
def test_infinite_first_diagonal_entry_deflates(gpu, n):
    # H(1, 0) is negligible beside an infinite H(0, 0): the others are the eigenvalues of the rest
    A = np.triu(H.gaussian(1, n, 9400 + n), -1)
    for k in range(1, n):
        A[0, k, k - 1] = abs(A[0, k, k - 1])
    want = np.linalg.eigvals(A[0, 1:, 1:])
    A[0, 0, 0] = np.inf
    h, z, e = planes(A), planes(np.eye(n)[None] + 0j), zeros(n)
    info = torch.full((1,), -1, dtype=torch.int32, device="cuda")
    veig.zlahqr(n, 1, 1, *e, *h, *z, info=info)
    assert int(info[0]) == 0
    _, err = H.match_eigenvalues(want[None], vec(e, n)[:, 1:])
    assert np.all(err <= 1e-11 * norm(A[:, 1:, 1:]))


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("n,m", [(n, m) for n in (33, 48, 64, 65, 80, 96) for m in (n // 2, 32, 24)] + [(16, 8), (24, 15)])
def test_deflated_block_beside_an_undefined_one(gpu, n, m, bad):
    # H(m, m-1) = 0: no rotation of the block from m on touches the columns
    # before it, in T and in Z, and the eigenvalues there are theirs
    A = np.triu(H.gaussian(1, n, 9500 + n), -1)
    for k in range(1, n):
        A[0, k, k - 1] = abs(A[0, k, k - 1])
    A[0, m, m - 1] = 0
    want = np.linalg.eigvals(A[0, :m, :m])
    for r, c in ((m, m), (n - 1, n - 1), (0, m), (m - 1, m)):
        B = A.copy()
        B[0, r, c] = bad
        h, z, e = planes(B), planes(np.eye(n)[None] + 0j), zeros(n)
        veig.zlahqr(n, 1, 1, *e, *h, *z)
        T, Z = back(h, n)[0], back(z, n)[0]
        _, err = H.match_eigenvalues(want[None], vec(e, n)[:, :m])
        assert np.all(err <= 1e-11 * norm(A[:, :m, :m]))
        assert np.all(np.tril(T, -1) == 0)
        R = A[0, :m, :m] @ Z[:m, :m] - Z[:m, :m] @ T[:m, :m]
        assert norm(R) <= 1e-13 * n * norm(A[0, :m, :m])
        assert np.all(Z[m:, :m] == 0)


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("n", [33, 48, 64, 65, 80, 96])
def test_schur_vectors_beside_an_undefined_column(gpu, n, bad):
    # diagonal but for one block: columns of Z outside it are copied
    m = n // 2
    A = np.diag(np.arange(1, n + 1) + 0j)[None].copy()
    A[0, m:m + 3, m:m + 3] = np.triu(H.gaussian(1, 3, 9600 + n)[0], -1)
    A[0, m + 1, m], A[0, m + 2, m + 1] = 1, 1
    Z0 = H.gaussian(1, n, 9700 + n)
    Z0[0, 0, m + 3], Z0[0, 1, m - 1], Z0[0, 2, n - 1], Z0[0, 3, m + 1] = bad, bad, bad, bad
    h, z, e = planes(A), planes(Z0), zeros(n)
    veig.zlahqr(n, 1, 1, *e, *h, *z)
    Z = back(z, n)[0]
    keep = np.r_[0:m, m + 3:n]
    finite = np.isfinite(Z0[0][:, keep])
    assert np.array_equal(Z[:, keep][finite], Z0[0][:, keep][finite])
    assert np.all(np.isfinite(np.delete(Z[:, m:m + 3], 3, axis=0)))
