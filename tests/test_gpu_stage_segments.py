"""The stage entries above order 80 on both segment widths of the Schur vectors
(24 and 48 columns to a lane): zlahqr on either side of four matrices per CU and
of the orders where two of its workgroups share a CU (89 / 90, 93 / 94), ztrevc."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
import veig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,N", [(81, 2), (81, 1026), (89, 2), (89, 1026), (90, 2), (93, 2), (94, 2), (96, 2), (96, 1026)])
def test_stages_above_80(gpu, n, N):
    A = np.tile(H.gaussian(2, n, 8600 + n), (N // 2, 1, 1))
    rH, iH = (torch.from_numpy(x).cuda() for x in H.to_soa(A, 2))
    rZ, iZ = torch.empty_like(rH), torch.empty_like(iH)
    rE, iE = (torch.empty(N * n, dtype=torch.float64, device="cuda") for _ in range(2))
    info = torch.full((N,), -1, dtype=torch.int32, device="cuda")
    back = lambda r, i: H.from_soa(r.cpu().numpy(), i.cpu().numpy(), n, 2)  # noqa: E731
    veig.hessenberg(n, N // 2, 2, rH, iH, rZ, iZ)
    veig.zlahqr(n, N // 2, 2, rE, iE, rH, iH, rZ, iZ, info=info)
    T, Z = np.triu(back(rH, iH)), back(rZ, iZ)
    E = H.vec_from_soa(rE.cpu().numpy(), iE.cpu().numpy(), n, 2)
    tol = 1e-13 * n
    assert int((info != 0).sum()) == 0
    for m in (slice(0, 2), slice(N - 2, N)):
        norm = np.linalg.norm(A[m], axis=(1, 2))
        assert np.all(np.linalg.norm(np.conj(np.swapaxes(Z[m], 1, 2)) @ Z[m] - np.eye(n), axis=(1, 2)) <= tol)
        assert np.all(np.linalg.norm(A[m] @ Z[m] - Z[m] @ T[m], axis=(1, 2)) <= tol * norm)
    veig.ztrevc(n, N // 2, 2, rH, iH, rZ, iZ)
    V = back(rZ, iZ)
    for m in (slice(0, 2), slice(N - 2, N)):
        assert np.all(H.backward_error(A[m], E[m], V[m]) <= 64 * n * np.finfo(float).eps)
