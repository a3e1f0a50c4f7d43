"""A NaN or an infinity reaches the rows that couple to it and no others, in
every kernel that reads narrow column ids (whose unused slots multiply another
row's x by 0) and in the reference-order panels.

A x is compared with the grid's neighbours; sweeps and V-cycles, where it
spreads on, with the 32-bit columns and the launches per hyperplane; and the
problems of a fleet keep it to themselves."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


@pytest.fixture(scope="module")
def hp():
    import torch
    assert torch.cuda.is_available()
    import hpcg_amd
    return hpcg_amd


def neighbours(g, dims):
    nx, ny, nz = dims
    x, y, z = g % nx, g // nx % ny, g // (nx * ny)
    return {(c * ny + b) * nx + a
            for c in range(max(0, z - 1), min(nz, z + 2))
            for b in range(max(0, y - 1), min(ny, y + 2))
            for a in range(max(0, x - 1), min(nx, x + 2))}


def places(dims, count=10):
    """Corners, and random rows of every kind."""
    nx, ny, nz = dims
    corners = [(c * ny + b) * nx + a
               for a, b, c in itertools.product((0, nx - 1), (0, ny - 1), (0, nz - 1))]
    rng = np.random.default_rng(nx * ny + nz)
    edge = [int(rng.integers(ny * nz)) * nx + int(rng.choice([0, nx - 1])) for _ in range(count)]
    return sorted(set(corners + edge + [int(g) for g in rng.integers(nx * ny * nz, size=count)]))


def bad_rows(P, y):
    return set(np.flatnonzero(~np.isfinite(P.to_numpy(y))).tolist())


GRIDS = [(16, 16, 16), (32, 32, 32), (64, 64, 8), (33, 31, 29), (20, 18, 13), (70, 33, 6)]


@pytest.mark.parametrize("stream", [0, 1])
@pytest.mark.parametrize("dims", GRIDS)
def test_spmv_reaches_neighbours_only(hp, dims, stream):
    import torch
    P = hp.Problem.generate(*dims, nlevels=1)
    if stream:
        P.tune("stream_min_bytes", 0)
    n = P.nrow(0)
    for k, g in enumerate(places(dims)):
        want = neighbours(g, dims)
        x = np.ones(n)
        x[g] = (NAN, INF, -INF)[k % 3]
        xd = P.to_device_order(x)
        y = P.zeros()
        P.spmv(xd, y)
        assert bad_rows(P, y) == want, g
        y32 = torch.zeros(n, dtype=torch.float32, device="cuda")
        P.spmv32(xd.float(), y32)
        assert bad_rows(P, y32.double()) == want, g
        X = torch.ones((n, 4), dtype=torch.float64, device="cuda")
        X[:, 2] = xd
        Y = torch.zeros_like(X)
        P.spmv_block(X, Y)
        assert bad_rows(P, Y[:, 2].contiguous()) == want, g
        assert Y[:, [0, 1, 3]].isfinite().all()
    P.close()


def same(a, b):
    import torch
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(
        a.nan_to_num(nan=0.5, posinf=INF, neginf=-INF), b.nan_to_num(nan=0.5, posinf=INF, neginf=-INF))


def sweeps(P, r, x):
    """Every sweep and V-cycle from r and x."""
    import torch
    out = []
    for order in ("multicolor", "lexicographic"):
        y = x.clone()
        P.symgs(r, y, ordering=order)
        z = torch.empty_like(r)
        P.mg(r, z, ordering=order)
        out += [y, z]
    y = x.float()
    P.symgs32(r.float(), y, ordering="multicolor")
    z = torch.empty_like(y)
    P.mg32(r.float(), z, ordering="multicolor")
    out += [y, z]
    for s in (2, 4, 8):
        R = torch.stack([r, r * 0.5, x, r - x] * 2, dim=1)[:, :s].float().contiguous()
        Z = torch.empty_like(R)
        P.mg32_block(R, Z, ordering="multicolor")
        out.append(Z)
    P.check()
    return out


@pytest.mark.parametrize("knobs", [{"zero_live": 11}, {"zero_live": 4}, {"zero_live": 0},
                                   {"col8": 0}, {"affine8": 0}, {"fp16_pairs": 0}, {"turn": 0},
                                   {"zero_guess": 0},
                                   {"x_pairs": 15, "block_pairs": 1, "stream_min_bytes": 0}])
@pytest.mark.parametrize("dims,levels", [((16, 16, 16), 2), ((32, 32, 32), 3), ((33, 31, 29), 1),
                                         ((36, 20, 28), 3), ((64, 64, 8), 2)])
def test_sweeps_as_by_32bit_columns(hp, dims, levels, knobs):
    import torch
    P = hp.Problem.generate(*dims, nlevels=levels)
    for key, value in knobs.items():
        P.tune(key, value)
    n = P.nrow(0)
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    r0, x0 = (torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
              for _ in range(2))
    for k, at in enumerate([0, n - 1, n // 3, dims[0] * dims[1] - 1]):
        at = int(P.to_device_order(np.arange(n) == at).argmax())
        r, x = r0.clone(), x0.clone()
        (r if k % 2 else x)[at] = (NAN, INF)[k // 2]
        outs = []
        for narrow in (1, 0):
            P.tune("col16", narrow)
            P.tune("tail", narrow)
            P.tune("lex_panels", narrow)
            outs.append(sweeps(P, r, x))
        for q, (a, b) in enumerate(zip(*outs)):
            assert same(a, b), (k, q)
    P.close()


@pytest.mark.parametrize("tail", [1, 0])
@pytest.mark.parametrize("dims", [((10, 12, 14), (9, 7, 11), (20, 10, 30)), ((16, 16, 16),) * 6,
                                  ((10, 10, 10),) * 8, ((16, 16, 16), (8, 16, 24), (24, 24, 24))])
def test_fleet_problems_apart(hp, dims, tail):
    import torch
    P = hp.Problem.generate_fleet(dims, nlevels=1)
    P.tune("tail", tail)
    n = P.nrow(0)
    offs = P.fleet_offsets()
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    r0, x0 = (torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
              for _ in range(2))
    clean = sweeps(P, r0, x0)
    for at in (0, offs[1] - 1, offs[1], offs[2] - 1, offs[-1] - 1, (offs[1] + offs[2]) // 2):
        q = int(np.searchsorted(offs, at, "right")) - 1
        row = int(P.to_device_order(np.arange(n) == at).argmax())
        own = P.to_device_order((np.arange(n) >= offs[q]) & (np.arange(n) < offs[q + 1])) > 0
        r, x = r0.clone(), x0.clone()
        r[row] = x[row] = NAN
        for k, (a, b) in enumerate(zip(sweeps(P, r, x), clean)):
            assert torch.equal(a[~own], b[~own]), (at, k)
    P.close()


def test_large_colour_steps(hp):
    """Colour steps of more than 6 * 2^20 rows (all else equal)."""
    import torch
    P = hp.Problem.generate(384, 376, 372, nlevels=1)
    n = P.nrow(0)
    r = torch.full((n,), 0.25, dtype=torch.float64, device="cuda")
    outs = []
    for narrow in (1, 0):
        P.tune("col16", narrow)
        x = torch.linspace(-1.0, 1.0, n, dtype=torch.float64, device="cuda")
        x[n // 2 + 17] = NAN
        P.symgs(r, x, ordering="multicolor")
        outs.append(x)
    assert outs[0].isfinite().any() and same(*outs)
    P.close()


@pytest.mark.parametrize("graph", [False, True])
def test_fleet_cg_apart(hp, graph):
    """A problem whose right-hand side holds a NaN is reported; the others'
    solutions are those they have without it."""
    import torch
    dims = ((10, 10, 10),) * 3 + ((16, 16, 16), (8, 16, 24))
    P = hp.Problem.generate_fleet(dims, nlevels=1)
    n = P.nrow(0)
    offs = P.fleet_offsets()
    b = P.to_device_order(np.random.default_rng(5).random(n) - 0.5)
    clean = torch.zeros_like(b)
    P.cg_fleet(b, clean, max_iter=4, graph=graph)
    b[int(P.to_device_order(np.arange(n) == offs[2] - 1).argmax())] = NAN
    x = torch.zeros_like(b)
    with pytest.raises(hp._lib.HpcgxError, match="not finite"):
        P.cg_fleet(b, x, max_iter=4, graph=graph)
    own = P.to_device_order((np.arange(n) >= offs[1]) & (np.arange(n) < offs[2])) > 0
    assert torch.equal(x[~own], clean[~own])
    P.close()
