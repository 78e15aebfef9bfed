"""Which wavefront runs the chain: every wavefront of a workgroup must name the
same one, also where their registers tell of different places (a workgroup that
was restored elsewhere between two reads), and neighbours on a CU name wavefronts
on different SIMDs."""
from __future__ import annotations

import ctypes
from pathlib import Path

import numpy as np
import pytest

LIB = Path(__file__).resolve().parent / "probe" / "libchain_probe_host.so"


def picks(simds, places, size=5):
    L = ctypes.CDLL(str(LIB))
    n = len(simds)
    hw = (ctypes.c_uint * n)(*[0x100 | s << 4 | 7 for s in simds])
    lds = (ctypes.c_uint * n)(*[p * size | size << 12 for p in places])
    out = (ctypes.c_int * n)()
    L.probe_chain(n, hw, lds, out)
    return list(out)


@pytest.mark.parametrize("waves", range(1, 9))
def test_one_choice(waves):
    rng = np.random.default_rng(waves)
    for _ in range(500):
        p = picks(rng.integers(0, 4, waves).tolist(), rng.integers(0, 8, waves).tolist())
        assert len(set(p)) == 1 and 0 <= p[0] < waves


def test_no_lds_size():
    assert len(set(picks([0, 1, 2, 3], [0] * 4, size=0))) == 1


def test_neighbours_on_different_simds():
    # four workgroups of three wavefronts, each SIMD left out once
    left_out = [[s for s in range(4) if s != o] for o in range(4)]
    assert sorted(g[picks(g, [0] * 3)[0]] for g in left_out) == [0, 1, 2, 3]
    # workgroups of four wavefronts, by their place
    assert sorted(picks([0, 1, 2, 3], [p] * 4)[0] for p in range(4)) == [0, 1, 2, 3]
