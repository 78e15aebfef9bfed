"""Uneven batches at the borders of the slot capacities (12, 16, 24, 28, 32), with
grids so small that every wavefront takes many sets of matrices, empty parts
among them, and chunks of the scatter that end inside a workgroup; against the
oracle, on two runs in a row and under capture."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import veig
from test_gpu_varsize import build, check_all, fetch

pytestmark = pytest.mark.gpu

PARTS = {
    "borders": [8, 9, 12, 13, 16, 17, 24, 25, 28, 29, 32],
    "no part in the middle": [20, 24, 30],
    "the middle alone": [25, 26, 28],
    "one order": [32],
}


@pytest.mark.parametrize("name", sorted(PARTS))
@pytest.mark.parametrize("grid", [0, 1, 3])
def test_parts_and_small_grids(gpu, name, grid):
    rng = np.random.default_rng(len(name))
    dims = rng.choice(PARTS[name], 263).tolist()
    vb, mats = build(dims, 5)
    if grid:
        vb.grid = [grid] * 5
    for _ in range(2):
        vb.rV.fill_(float("nan"))
        vb.info.fill_(-7)
        vb.run()
        torch.cuda.synchronize()
        check_all(mats, fetch(vb, dims), vb.info.cpu().numpy(), dims)
    g = vb.graph()
    vb.rV.fill_(float("nan"))
    for _ in range(2):
        g.launch()
    torch.cuda.synchronize()
    check_all(mats, fetch(vb, dims), vb.info.cpu().numpy(), dims)
