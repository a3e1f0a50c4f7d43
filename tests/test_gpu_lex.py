"""Reference-order sweeps by panels of rows (lex.hip): the same bits as one
launch per hyperplane, which test_gpu_parity.py compares with the oracle.

Sizes: a few rows; planes whose hyperplanes hold fewer rows than a wavefront,
several wavefronts, and more than a workgroup takes in one step; one plane;
one line; a fleet (planes of several grids); a host matrix with no grid
dimensions (panels as wide as the matrix; one panel); a random diagonal and a
matrix whose rows store zeros (32-bit columns)."""
import numpy as np
import pytest

from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hp():
    import torch
    assert torch.cuda.is_available()
    import hpcg_amd
    return hpcg_amd


def host_levels(dims, grid, zeros=False):
    h = O.Hierarchy(*dims, nlevels=1)
    m = h.level(0)
    d = {k: np.array(m[k]) for k in ("nnz_row", "cols", "vals", "diag_slot")}
    if zeros:  # every seventh row stores a zero off the diagonal
        v = d["vals"].reshape(-1, 27)
        first = np.where(d["diag_slot"] == 0, 1, 0)
        rows = np.arange(0, v.shape[0], 7)
        v[rows, first[rows]] = 0.0
        d["vals"] = v.reshape(-1)
    d.update(zip(("nx", "ny", "nz"), dims if grid else (0, 0, 0)))
    return [d]


def both(P, level=0, seed=0, mg=False):
    """x after one sweep (or V-cycle) by panels and by hyperplanes."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n = P.nrow(level)
    r, x = (torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
            for _ in range(2))
    out = []
    for on in (1, 0):
        P.tune("lex_panels", on)
        y = x.clone()
        if mg:
            P.mg(r, y, ordering="lexicographic")
        else:
            P.symgs(r, y, level=level, ordering="lexicographic")
        P.check()
        out.append(y)
    P.tune("lex_panels", 1)
    return out


CASES = [("grid", d) for d in ((1, 1, 3), (2, 2, 2), (5, 1, 1), (7, 5, 9), (64, 40, 1),
                               (33, 130, 6), (70, 64, 12), (700, 640, 3))]
CASES += [("fleet", ((8, 8, 16), (24, 8, 8), (16, 40, 8))),
          ("nogrid", (12, 10, 9)), ("nogrid", (60, 48, 40)), ("zeros", (20, 18, 11))]


@pytest.mark.parametrize("kind,dims", CASES)
def test_lex_panels_same_bits(hp, kind, dims):
    import torch
    print("[case]", kind, dims, flush=True)
    if kind == "fleet":
        P = hp.Problem.generate_fleet(dims, nlevels=4)
    elif kind == "grid":
        P = hp.Problem.generate(*dims, nlevels=1)
    else:
        P = hp.Problem.from_reference_levels(host_levels(dims, False, kind == "zeros"))
    for l in range(P.nlevels):
        a, b = both(P, l, seed=l)
        assert torch.equal(a, b), l
    d = P.copy_diagonal() * (1.0 + torch.rand(P.nrow(0), dtype=torch.float64, device="cuda"))
    P.replace_diagonal(d)  # the copy follows
    a, b = both(P, seed=7)
    assert torch.equal(a, b)
    P.close()


def test_lex_panels_streams_and_capture(hp):
    """Sweeps on two streams share the copy's scratch in turn; a sweep under a
    caller's capture replays with the same bits."""
    import torch
    P = hp.Problem.generate(32, 24, 16, nlevels=3)
    want, _ = both(P, seed=1, mg=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    r, x = (torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
            for _ in range(2))
    refs = []
    for k in range(4):
        y = x * (k + 1)
        P.symgs(r, y, ordering="lexicographic")
        refs.append(y)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [x * (k + 1) for k in range(4)]
    torch.cuda.synchronize()
    for k in range(4):
        with torch.cuda.stream(streams[k % 2]):
            P.symgs(r, got[k], ordering="lexicographic")
    torch.cuda.synchronize()
    for a, b in zip(refs, got):
        assert torch.equal(a, b)
    z = torch.zeros_like(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        P.mg(r, z, ordering="lexicographic")
    for _ in range(3):
        z.fill_(5.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, want)
        P.mg(r, x.clone(), ordering="lexicographic")  # eager work in between
    P.close()
