"""The one-matrix-per-workgroup kernels (veig_stream.hpp: orders 33..96) at the
edges of their capacities (48, 64, 80, 96 for the reduction; segments of 20, 24
and 32 columns for the Schur vectors) and on inputs that take their rare
branches, against the oracle at the bar of test_gpu_parity."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
import veig
from gpu_util import gpu_eig
from test_gpu_parity import check_parity, constructed

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n", [33, 40, 41, 48, 49, 64, 65, 80, 81, 96])
def test_capacity_edges(gpu, n):
    A = H.gaussian(3, n, 4000 + n)
    E, V, info, T = gpu_eig(A, 3 if n % 2 else 1, write_schur=True)
    Eo, Vo, _ = H.oracle_eig(A, 3 if n % 2 else 1)
    check_parity(A, E, V, info, Eo, Vo)
    assert np.max(np.abs(np.tril(T, -1))) == 0.0
    assert np.allclose(np.diagonal(T, axis1=1, axis2=2), E, atol=0)


@pytest.mark.parametrize("n", [33, 57, 64])
def test_eigenvalues_only_edges(gpu, n):
    A = H.gaussian(5, n, 4100 + n)
    rA, iA = (torch.from_numpy(x).cuda() for x in H.to_soa(A, 5))
    rE, iE = veig.eigvals(rA, iA, n, 1, 5)
    E = H.vec_from_soa(rE.cpu().numpy(), iE.cpu().numpy(), n, 5)
    Eo, _, _ = H.oracle_eig(A, 5)
    _, err = H.match_eigenvalues(Eo, E)
    assert np.all(err <= 1e-11 * np.linalg.norm(A, axis=(1, 2)))


@pytest.mark.parametrize("n", [34, 66])
def test_deflated_and_undefined_inputs_beside_ordinary_ones(gpu, n):
    # no sweep at all (zero, diagonal, triangular), a cyclic permutation
    # (exceptional shifts), entries of 1e150, NaN: each ends, and none changes
    # its neighbours
    G = H.gaussian(2, n, 4200 + n)
    cyc = np.roll(np.eye(n), 1, axis=0).astype(complex)
    tri = np.triu(H.gaussian(1, n, 4300 + n)[0]) + np.diag(np.arange(n) * 3.0)
    nan = np.full((n, n), np.nan + 0j)
    A = np.stack([G[0], np.zeros((n, n), complex), np.diag(np.arange(1, n + 1) + 0j), tri, cyc, G[1] * 1e150, nan,
                  G[1]])
    E, V, info = gpu_eig(A, 1)
    alone, _, _ = gpu_eig(G, 1)
    assert np.array_equal(E[0], alone[0]) and np.array_equal(E[7], alone[1])
    assert np.all(info[[0, 1, 2, 3, 5, 7]] == 0)
    assert np.all(E[1] == 0)
    for m in (2, 3):
        assert np.allclose(np.sort_complex(E[m]), np.sort_complex(np.diag(A[m])), atol=1e-12 * n)
    if info[4] == 0:
        assert np.allclose(np.abs(E[4]), 1.0, atol=1e-12 * n)
    _, err = H.match_eigenvalues(E[7:8], E[5:6] / 1e150)
    assert np.all(err <= 1e-11 * np.linalg.norm(G[1]))
    assert not np.any(np.isfinite(E[6]))


@pytest.mark.parametrize("n", [40, 60])
def test_mixed_list_solves(gpu, n):
    # cond(V) = 1e7: complex64 does not reach the tolerance, so the listed
    # matrices are solved again in FP64
    A = np.concatenate([constructed(3, n, 44, cond=1e7), H.gaussian(2, n, 45)])
    rA, iA = (torch.from_numpy(x).cuda() for x in H.to_soa(A, 1))
    fb = torch.full((5,), -1, dtype=torch.int32, device="cuda")
    berr = torch.zeros(5, dtype=torch.float64, device="cuda")
    rE, iE, rV, iV = veig.zgeev_mixed(rA, iA, n, 5, 1, fallback=fb, berr=berr)
    E = H.vec_from_soa(rE.cpu().numpy(), iE.cpu().numpy(), n, 1)
    V = H.from_soa(rV.cpu().numpy(), iV.cpu().numpy(), n, 1)
    assert np.all(fb.cpu().numpy()[:3] == 1)
    assert np.all(berr.cpu().numpy() <= 1e-12)
    assert np.all(H.backward_error(A, E, V) <= 1e-12)
