"""The measured work: batched complex eigenproblems through the package's
device entry points (`veig`), at the sizes of the repository's own
configurations (bench.py, workloads.py, tests/) and at odd ones between them.

A pass ends the way a program that stores or compares eigenvectors ends it:
the split planes become complex tensors, and every eigenvector is turned so
that its first component is real and positive.  The phase of a computed
eigenvector carries no information -- it is that of a subdiagonal entry which
was about to be dropped as negligible, so one unit in the last place of the
input turns it -- while its length (the eigenvector has a 1 at its own index
in the Schur basis) and the order of the eigenvalues (the order in which they
deflate) belong to the interface and are returned as they are.

Kinds of case (sizes: `n` the order, `batch` matrices in tiles of `tile`):
  solve    veig.zgeev, FP64: eigenvalues and eigenvectors
  mixed    veig.zgeev_mixed: complex64 solve refined in FP64
  values   veig.eigvals, FP64: eigenvalues only
  roots    veig.roots: polynomials of degree n by their companion matrices
  uneven   veig.VarBatch: orders lo..hi in one batch (`lo`, `hi`)
  stages   veig.hessenberg, veig.zlahqr, veig.ztrevc one after the other, as
           a program does that wants the Schur form too
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "vectorized-eigensolver_amd"))
import veig  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # a handful of matrices, as an interactive program or a test has them:
        # one matrix's latency and the launches
        dict(name="solve_16_few", kind="solve", n=16, batch=64, tile=4),
        # the smallest of the repository's configurations
        dict(name="solve_8_small", kind="solve", n=8, batch=4096, tile=64),
        # the headline configuration
        dict(name="solve_16_large", kind="solve", n=16, batch=1 << 20, tile=64),
        # an odd order in odd tiles
        dict(name="solve_27_ragged", kind="solve", n=27, batch=1501 * 13, tile=13),
        # the largest configuration, one matrix after another in memory
        dict(name="solve_64_large", kind="solve", n=64, batch=1 << 16, tile=1),
        # an order from the upper end of the reference driver's sweep
        dict(name="solve_79", kind="solve", n=79, batch=3328, tile=64),
        # stability analysis: eigenvalues without eigenvectors
        dict(name="values_48", kind="values", n=48, batch=1 << 14, tile=64),
        # polynomial roots at the repository's configuration
        dict(name="roots_16_large", kind="roots", n=16, batch=1 << 20, tile=64),
        # matrices of many orders in one call
        dict(name="uneven_4_32", kind="uneven", lo=4, hi=32, batch=1 << 17),
        # mixed precision on the headline batch
        dict(name="mixed_16_large", kind="mixed", n=16, batch=1 << 20, tile=64),
        # mixed precision at an order above 32
        dict(name="mixed_50", kind="mixed", n=50, batch=1 << 13, tile=8),
        # the stage entries one by one
        dict(name="stages_40", kind="stages", n=40, batch=1 << 11, tile=32),
    ]


# the most matrices a drawn case may hold at order n: its pass is shorter than
# that of the largest listed case
def _most(kind, n):
    flops = {"solve": 1.5e11, "mixed": 1.5e11, "values": 5e10, "roots": 5e10, "stages": 1e10}[kind]
    if n > 64:
        flops = 6e10
    return max(16, min(1 << 20, int(flops / _flops(kind, n))))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve"] * 5 + ["mixed", "mixed", "values", "values", "roots", "uneven", "stages"])
    if kind == "uneven":
        lo = rng.randint(2, 12)
        return dict(kind=kind, lo=lo, hi=rng.randint(lo + 1, 32), batch=_log(rng, 500, 1 << 17))
    top = {"solve": 96, "stages": 96}.get(kind, 64)
    n = rng.randint(4, top) if rng.random() < 0.7 else rng.choice([8, 16, 24, 32, 48, 64])
    tile = rng.choice([1, 4, 7, 13, 16, 32, 64])
    most = _most(kind, n)
    blocks = max(1, _log(rng, min(16, most), most) // tile)
    return dict(kind=kind, n=n, batch=blocks * tile, tile=tile)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _randn(count, g):
    return torch.randn(count, dtype=torch.float64, device=DEV, generator=g)


def prepare(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    kind, N = case["kind"], case["batch"]
    if kind == "uneven":
        return _prepare_uneven(case, g)
    n, tile = case["n"], case["tile"]
    s = dict(kind=kind, n=n, bc=N // tile, tc=tile)
    empty = lambda count: torch.empty(count, dtype=torch.float64, device=DEV)  # noqa: E731
    if kind == "roots":
        # coefficients c_0 .. c_n, iid complex Gaussian
        s["rC"], s["iC"] = _randn(N * (n + 1), g), _randn(N * (n + 1), g)
        return s
    # entries iid complex Gaussian (the layout does not matter for iid entries)
    s["rA"], s["iA"] = _randn(N * n * n, g), _randn(N * n * n, g)
    s["info"] = torch.empty(N, dtype=torch.int32, device=DEV)
    if kind == "stages":
        return s
    s["out"] = (empty(N * n), empty(N * n))
    if kind != "values":
        s["out"] += (empty(N * n * n), empty(N * n * n))
    if kind == "mixed":
        s["ws"] = veig.mixed_workspace(n, s["bc"], tile, DEV)
    return s


def _prepare_uneven(case, g):
    """Orders uniform in lo..hi (the same ones for every seed: a program that
    calls again has other matrices of the same orders), entries iid complex
    Gaussian.  Hermitian matrices are left out: the order in which their
    eigenvalues deflate is decided by rounding for one in a few thousand."""
    N = case["batch"]
    orders = torch.Generator()
    orders.manual_seed(1000 * case["lo"] + case["hi"])
    dims = torch.randint(case["lo"], case["hi"] + 1, (N,), generator=orders)
    vb = veig.VarBatch(dims)
    vb.rA.copy_(_randn(vb.total_a, g))
    vb.iA.copy_(_randn(vb.total_a, g))
    # the first entry of each entry's column, for the eigenvectors' phase
    dims = dims.to(DEV)
    mat = torch.repeat_interleave(torch.arange(N, device=DEV), dims * dims)
    local = torch.arange(vb.total_a, device=DEV) - vb.a_off[mat]
    return dict(kind="uneven", vb=vb, first=vb.a_off[mat] + local // dims[mat] * dims[mat])


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _vectors(rV, iV, n, bc, tc):
    """The eigenvectors as a complex tensor [block, column, row, matrix], the
    first component of each real and positive."""
    V = torch.complex(rV, iV).view(bc, n, n, tc)
    return V.mul_(torch.sgn(V[:, :, :1, :]).conj())


def run(s):
    kind = s["kind"]
    if kind == "uneven":
        vb = s["vb"]
        vb.run()
        V = torch.complex(vb.rV, vb.iV)
        return dict(E=torch.complex(vb.rE, vb.iE), V=V * torch.sgn(V[s["first"]]).conj(), info=vb.info)
    n, bc, tc = s["n"], s["bc"], s["tc"]
    if kind == "roots":
        rE, iE = veig.roots(s["rC"], s["iC"], n, bc, tc)
        return dict(E=torch.complex(rE, iE))
    if kind == "values":
        rE, iE = veig.eigvals(s["rA"], s["iA"], n, bc, tc, out=s["out"], info=s["info"])
        return dict(E=torch.complex(rE, iE), info=s["info"])
    if kind == "stages":
        return _run_stages(s, n, bc, tc)
    if kind == "mixed":
        rE, iE, rV, iV = veig.zgeev_mixed(s["rA"], s["iA"], n, bc, tc, out=s["out"], info=s["info"],
                                          workspace=s["ws"])
    else:
        rE, iE, rV, iV = veig.zgeev(s["rA"], s["iA"], n, bc, tc, out=s["out"], info=s["info"])
    return dict(E=torch.complex(rE, iE), V=_vectors(rV, iV, n, bc, tc), info=s["info"])


def _run_stages(s, n, bc, tc):
    rH, iH = s["rA"].clone(), s["iA"].clone()          # the stages work in place
    rZ, iZ = torch.empty_like(rH), torch.empty_like(iH)
    veig.hessenberg(n, bc, tc, rH, iH, rZ, iZ)          # H, Q
    rE, iE = (torch.empty(bc * tc * n, dtype=torch.float64, device=rH.device) for _ in range(2))
    veig.zlahqr(n, bc, tc, rE, iE, rH, iH, rZ, iZ, info=s["info"])  # T, Z
    # the Schur vectors' phases, from their first components
    first = lambda p: p.view(bc, n, n, tc)[:, :, 0, :]  # noqa: E731
    d = torch.sgn(torch.complex(first(rZ), first(iZ))).conj()       # [block, column, matrix]
    T = torch.complex(rH, iH).view(bc, n, n, tc)                    # [block, column, row, matrix]
    T = T * d.unsqueeze(2) * d.conj().unsqueeze(1)
    veig.ztrevc(n, bc, tc, rH, iH, rZ, iZ)                          # V over Z
    return dict(E=torch.complex(rE, iE), T=T, V=_vectors(rZ, iZ, n, bc, tc), info=s["info"])


def exact(case, seed):
    """Nothing here has a value of its own in 64 bits: the order in which the
    eigenvalues of a matrix are found, and with it the length of every
    eigenvector, is the iteration's, and no library's iteration shares it."""
    return None


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _flops(kind, n):
    """Per matrix, as bench.py counts them: the Hessenberg reduction, the
    unitary factor, two QR sweeps per eigenvalue and the eigenvectors (complex
    multiply-add = 8)."""
    gehrd = sum(16 * n * k + 16 * k * k for k in range(1, n))
    unghr = sum(16 * m * (m - 1) for m in range(1, n))
    trevc = sum(4 * (k - 1) ** 2 + 8 * n * (k - 1) for k in range(2, n + 1))
    qr = 20 * (2 * n + 3) * n * (n - 1)
    qr_values = sum(40 * (m + 3) * (m - 1) for m in range(2, n + 1))
    if kind == "roots":
        return qr_values
    if kind == "values":
        return gehrd + qr_values
    return gehrd + unghr + qr + trevc


def work(case):
    kind, N = case["kind"], case["batch"]
    if kind == "uneven":
        orders = range(case["lo"], case["hi"] + 1)
        flops = sum(_flops("solve", n) for n in orders) / len(orders)
        size = sum(32 * n * n + 16 * n for n in orders) / len(orders)
        return {"bytes": N * size, "flops": N * flops}
    n = case["n"]
    size = {"roots": 16 * (n + 1) + 16 * n, "values": 16 * n * n + 16 * n,
            "stages": 48 * n * n + 16 * n}.get(kind, 32 * n * n + 16 * n)
    return {"bytes": float(N * size), "flops": float(N * _flops(kind, n))}
