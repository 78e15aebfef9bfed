"""The per-matrix entries of veig_compat.hpp beside batches of every size: the
kernels that a batch takes depend on how many matrices it has, and a slot takes
its batch's, so the values stay the batch entry's to the bit (test_gpu_slots has
one size)."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import helpers as H
import veig

pytestmark = pytest.mark.gpu
DP = ctypes.POINTER(ctypes.c_double)
TC = 4


def fn(name, argtypes):
    f = getattr(veig.lib(), name)
    f.argtypes = argtypes
    f.restype = None
    return f


def at(a, off):
    return ctypes.cast(a.ctypes.data + 8 * off, DP)


def slot_of(a, b, t, size):
    return a[b * TC * size + t:][:size * TC:TC]


@pytest.mark.parametrize("n,bc", [(8, 64), (8, 257), (13, 256), (13, 257), (16, 257), (17, 257), (32, 257), (48, 3)])
def test_reduction(gpu, n, bc):
    rA, iA = H.to_soa(np.tile(H.gaussian(TC, n, 3101), (bc, 1, 1)), TC)
    rt, it = np.zeros(bc * TC * n), np.zeros(bc * TC * n)
    r0, i0 = rA.copy(), iA.copy()
    fn("_Z11test_zgehrdPdS_S_S_S_S_iii", [DP] * 6 + [ctypes.c_int] * 3)(*map(H.dptr, (rA, iA, rt, it)), None, None, n, bc, TC)
    rQ, iQ = rA.copy(), iA.copy()
    fn("_Z11test_zunghrPdS_S_S_S_S_iii", [DP] * 6 + [ctypes.c_int] * 3)(*map(H.dptr, (rQ, iQ, rt, it)), None, None, n, bc, TC)
    for b, t in ((0, 0), (bc - 1, 2)):
        mo, vo = b * TC * n * n + t, b * TC * n + t
        s, si, u, ui = r0.copy(), i0.copy(), np.zeros_like(rt), np.zeros_like(it)
        p = (at(s, mo), at(si, mo), at(u, vo), at(ui, vo), None, None, n, bc, TC)
        fn("_Z6zgehrdPdS_S_S_S_S_iii", [DP] * 6 + [ctypes.c_int] * 3)(*p)
        for x, y, size in ((s, rA, n * n), (si, iA, n * n), (u, rt, n), (ui, it, n)):
            assert np.array_equal(slot_of(x, b, t, size), slot_of(y, b, t, size))
        fn("_Z6zunghrPdS_S_S_S_S_iii", [DP] * 6 + [ctypes.c_int] * 3)(*p)
        for x, y in ((s, rQ), (si, iQ)):
            assert np.array_equal(slot_of(x, b, t, n * n), slot_of(y, b, t, n * n))


@pytest.mark.parametrize("n,bc", [(8, 64), (8, 65), (16, 65), (17, 65), (27, 65), (32, 65), (40, 3), (65, 129), (80, 129),
                                  (81, 257), (89, 3), (94, 3)])
def test_qr_and_eigenvectors(gpu, n, bc):
    rV, iV = H.to_soa(np.tile(H.hessenberg_input(TC, n, 3102), (bc, 1, 1)), TC)
    rZ, iZ = H.to_soa(np.tile(np.eye(n)[None] + 0j, (bc * TC, 1, 1)), TC)
    rE, iE = np.zeros(bc * TC * n), np.zeros(bc * TC * n)
    start = [x.copy() for x in (rV, iV, rE, iE, rZ, iZ)]
    fn("_Z10zlahqr_newPdS_S_S_S_S_iiii", [DP] * 6 + [ctypes.c_int] * 4)(*map(H.dptr, (rE, iE, rV, iV, rZ, iZ)), n, n * n, bc, TC)
    rR, iR = rZ.copy(), iZ.copy()
    fn("_Z11test_ztrevcPdS_S_S_S_S_iiii", [DP] * 6 + [ctypes.c_int] * 4)(*map(H.dptr, (rV, iV, rR, iR)), None, None, n, n * n, bc, TC)
    for b, t in ((0, 1), (bc - 1, 3)):
        mo, vo = b * TC * n * n + t, b * TC * n + t
        v, vi, e, ei, z, zi = (x.copy() for x in start)
        fn("_Z12zlahqr_schurbbiPdS_S_S_S_S_ii", [ctypes.c_bool, ctypes.c_bool, ctypes.c_int] + [DP] * 6 + [ctypes.c_int] * 2)(
            True, True, n, at(v, mo), at(vi, mo), at(e, vo), at(ei, vo), at(z, mo), at(zi, mo), bc, TC)
        for x, y, size in ((v, rV, n * n), (vi, iV, n * n), (e, rE, n), (ei, iE, n), (z, rZ, n * n), (zi, iZ, n * n)):
            assert np.array_equal(slot_of(x, b, t, size), slot_of(y, b, t, size))
        fn("_Z6ztrevcPdS_S_S_S_S_S_S_iii", [DP] * 8 + [ctypes.c_int] * 3)(
            at(v, mo), at(vi, mo), None, None, at(z, mo), at(zi, mo), None, None, n, bc, TC)
        for x, y in ((z, rR), (zi, iR)):
            assert np.array_equal(slot_of(x, b, t, n * n), slot_of(y, b, t, n * n))
