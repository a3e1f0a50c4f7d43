"""Workloads of the PCG path for timing: what they run, their compulsory work and their 64-bit results.

Every case goes through hpcg_amd.Problem as a program that solves with it does: the problem is
generated once (`prepare`), then whole calls are made on it (`run`).  Kinds:

  cg      FP64 PCG with the 4-level multigrid V-cycle (multicolour smoother)
  mixed   PCG with the FP32 V-cycle on FP16 matrix values, FP64 outside
  block   the mixed PCG for s right-hand sides at once
  fleet   independent problems on grids of their own, advanced together
  mg      one V-cycle in the reference's row order (lexicographic smoother)
  symgs   one symmetric multicolour smoother sweep of a single level
"""
import math

import torch

import hpcg_amd

# Position of greedy colour (x & 1) + 2 (y & 1) + 4 (z & 1) in the default sweep: device rows are
# sorted by it, in natural order inside a colour.
_SWEEP = (3, 5, 6, 7, 1, 2, 4, 0)


def listed():
    return [
        # the smallest configuration (16^3): a step's launches are all there is to it
        dict(name="cg-16", kind="cg", nx=16, ny=16, nz=16, levels=4, its=10, graph=True),
        # an odd-sized single level, no extent a multiple of anything: the smoother alone
        dict(name="symgs-151x133x97", kind="symgs", nx=151, ny=133, nz=97, levels=1),
        # the reference's row order on a small grid: hundreds of tiny dependent steps
        dict(name="mg-lex-64x48x32", kind="mg", nx=64, ny=48, nz=32, levels=4),
        # the reference's row order at the 256^3 configuration (the level-scheduled smoother)
        dict(name="mg-lex-256", kind="mg", nx=256, ny=256, nz=256, levels=4),
        # a mid-sized grid that is no power of two, launched call by call
        dict(name="cg-104x88x120", kind="cg", nx=104, ny=88, nz=120, levels=4, its=10, graph=False),
        # the 256^3 FP64 configuration
        dict(name="cg-256", kind="cg", nx=256, ny=256, nz=256, levels=4, its=6, graph=True),
        # FP64 on a grid near the benchmark-valid sizes: the largest
        dict(name="cg-512", kind="cg", nx=512, ny=512, nz=512, levels=4, its=3, graph=True),
        # mixed precision at 256^3, past one FP64 recompute of the residual
        dict(name="mixed-256", kind="mixed", nx=256, ny=256, nz=256, levels=4, its=11),
        # mixed precision at a large grid
        dict(name="mixed-384x448x416", kind="mixed", nx=384, ny=448, nz=416, levels=4, its=6),
        # block PCG at its 256^3 configuration
        dict(name="block-256-s8", kind="block", nx=256, ny=256, nz=256, levels=4, its=5, s=8),
        # block PCG with 16 right-hand sides on a ragged mid-sized grid
        dict(name="block-136x120x104-s16", kind="block", nx=136, ny=120, nz=104, levels=4, its=6,
             s=16),
        # the 32-problem fleet drawn from seed 7
        dict(name="fleet-32", kind="fleet", count=32, fleet_seed=7, levels=4, its=10),
    ]


def _extents(rng, lo, hi, step):
    """Three extents whose product is spread over its logarithm between lo and hi points, the
    aspect ratio over about a factor of two each way, each a multiple of `step`."""
    edge = math.exp(rng.uniform(math.log(lo), math.log(hi))) ** (1.0 / 3.0)
    a, b = (math.exp(rng.uniform(-0.35, 0.35)) for _ in range(2))
    return [max(2 * step, int(round(edge * f / step)) * step) for f in (a, b, 1.0 / (a * b))]


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "mixed", "mixed", "block", "fleet", "mg", "symgs"])
    if kind == "fleet":
        return dict(kind=kind, count=rng.randint(4, 40), fleet_seed=rng.randrange(1000), levels=4,
                    its=rng.randint(4, 10))
    if kind == "symgs":  # any extents, odd ones among them
        nx, ny, nz = _extents(rng, 2e4, 8e6, 1)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, levels=1)
    levels = rng.choice([3, 4, 4, 4])
    top = {"cg": 1.0e8, "mixed": 8e7, "block": 1.2e7, "mg": 1.4e7}[kind]
    low = {"cg": 4e3, "mixed": 1e5, "block": 5e4, "mg": 4e3}[kind]
    nx, ny, nz = _extents(rng, low, top, 2 ** (levels - 1))
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, levels=levels)
    if kind == "cg":
        case.update(its=rng.randint(3, 4), graph=rng.random() < 0.6)
    elif kind == "mixed":
        case.update(its=rng.choice([6, 8, 11]))
    elif kind == "block":
        case.update(its=rng.randint(3, 6), s=rng.choice([4, 8, 16]))
    return case


def _dims(case):
    if case["kind"] == "fleet":
        return hpcg_amd.fleet_dims(case["count"], case["fleet_seed"])
    return [(case["nx"], case["ny"], case["nz"])]


def _uniform(case, seed, which, columns=None):
    """uniform(-1, 1) values of the fine level in device row order, from the seed alone."""
    n = sum(a * b * c for a, b, c in _dims(case))
    where = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=where)
    g.manual_seed(2 * int(seed) + which)
    shape = (n,) if columns is None else (n, columns)
    return torch.rand(shape, generator=g, dtype=torch.float64, device=where).mul_(2.0).sub_(1.0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fleet":
        p = hpcg_amd.Problem.generate_fleet(_dims(case), nlevels=case["levels"])
    else:
        p = hpcg_amd.Problem.generate(case["nx"], case["ny"], case["nz"], nlevels=case["levels"])
    b = _uniform(case, seed, 0, case["s"] if kind == "block" else None)
    if kind == "mixed":
        p.prepare_mixed()
    # the smoother starts from some iterate, the solvers from 0, the V-cycle overwrites x
    x = _uniform(case, seed, 1) if kind == "symgs" else torch.zeros_like(b)
    return dict(case=case, p=p, b=b, x=x)


def run(state):
    case, p, b, x = state["case"], state["p"], state["b"], state["x"]
    kind = case["kind"]
    if kind == "symgs":
        p.symgs(b, x, level=0, ordering="multicolor")
        return x
    if kind == "mg":
        p.mg(b, x, level=0, ordering="lexicographic")
        return x
    x.zero_()
    if kind == "cg":
        r = p.cg(b, x, max_iter=case["its"], graph=case["graph"])
    elif kind == "mixed":
        r = p.cg_mixed(b, x, max_iter=case["its"], recompute=10)
    elif kind == "block":
        r = p.cg_block_mixed(b, x, max_iter=case["its"], recompute=10)
    else:
        r = p.cg_fleet(b, x, max_iter=case["its"], graph=True)
    return dict(x=x, niters=r["niters"] if kind != "fleet" else sum(r["niters"]),
                normr=torch.tensor(r["normr"], dtype=torch.float64),
                normr0=torch.tensor(r["normr0"], dtype=torch.float64))


# ---- compulsory work ---------------------------------------------------------------------------
def _grid_work(case, nx, ny, nz):
    """(bytes, flops) of one pass on one grid.  Each kernel of an iteration reads its matrix values
    once (column ids are the plan's to encode and are left out) and its vectors once."""
    kind, s = case["kind"], case.get("s", 1)
    val, vec = (2, 4) if kind in ("mixed", "block") else (8, 8)  # the smoother's storage

    def level(l):
        a, b, c = nx >> l, ny >> l, nz >> l
        return a * b * c, (3 * a - 2) * (3 * b - 2) * (3 * c - 2)

    n0, m0 = level(0)
    if kind == "symgs":
        return 2 * val * m0 + 6 * vec * n0, 4 * m0
    by = fl = 0
    for l in range(case["levels"]):
        n, m = level(l)
        sweeps = 2 if l + 1 < case["levels"] else 1
        by += sweeps * (2 * val * m + 6 * vec * n * s)
        fl += sweeps * 4 * m * s
        if l + 1 < case["levels"]:
            inj = ((3 * (nx >> l) // 2 - 1) * (3 * (ny >> l) // 2 - 1) * (3 * (nz >> l) // 2 - 1))
            nc = level(l + 1)[0]
            by += val * inj + (vec * n + 5 * vec * nc) * s
            fl += 2 * inj * s
    if kind == "mg":
        return by, fl
    # the outer product, its vectors (p, x, r updates) and dots in FP64
    by += val * m0 + (2 + 10) * 8 * n0 * s
    fl += (2 * m0 + 12 * n0) * s
    return by * case["its"], fl * case["its"]


def work(case):
    got = [_grid_work(case, *d) for d in _dims(case)]
    return dict(bytes=sum(g[0] for g in got), flops=sum(g[1] for g in got))


# ---- the same computation in plain torch, 64 bits ------------------------------------------------
def _box(x):
    """Sum over each point's 3 x 3 x 3 neighbourhood (grid in the last three axes)."""
    for d in (-1, -2, -3):
        y = x.clone()
        k = x.shape[d]
        y.narrow(d, 0, k - 1).add_(x.narrow(d, 1, k - 1))
        y.narrow(d, 1, k - 1).add_(x.narrow(d, 0, k - 1))
        x = y
    return x


def _apply(x):
    return 27.0 * x - _box(x)


def _colour_sweep(r, x):
    for c in _SWEEP + _SWEEP[::-1]:
        at = (Ellipsis, slice(c >> 2, None, 2), slice((c >> 1) & 1, None, 2), slice(c & 1, None, 2))
        x[at] = (r[at] + _box(x)[at] - x[at]) / 26.0


def _lex_sweep(r, x):
    """Natural-order sweep, hyperplane by hyperplane of x + 2y + 4z."""
    nz, ny, nx = r.shape
    pad = torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1))
    sy, sz = nx + 2, (nx + 2) * (ny + 2)
    z, y, i = torch.meshgrid(*(torch.arange(k, device=r.device) for k in (nz, ny, nx)),
                             indexing="ij")
    plane, order = torch.sort((i + 2 * y + 4 * z).reshape(-1), stable=True)
    cell = ((z + 1) * sz + (y + 1) * sy + i + 1).reshape(-1)[order]
    rhs, flat = r.reshape(-1)[order], pad.view(-1)
    near = torch.tensor([a * sz + b * sy + c for a in (-1, 0, 1) for b in (-1, 0, 1)
                         for c in (-1, 0, 1) if (a, b, c) != (0, 0, 0)], device=r.device)
    ends = torch.cumsum(torch.bincount(plane), 0).tolist()
    steps = list(zip([0] + ends[:-1], ends))
    for lo, hi in steps + steps[::-1]:
        at = cell[lo:hi]
        flat[at] = (rhs[lo:hi] + flat[at[:, None] + near].sum(1)) / 26.0
    x.copy_(pad[1:-1, 1:-1, 1:-1])


def _vcycle(r, levels, sweep):
    x = torch.zeros_like(r)
    sweep(r, x)
    if levels > 1:
        even = (Ellipsis,) + (slice(None, None, 2),) * 3
        coarse = (r - _apply(x))[even].contiguous()
        x[even] += _vcycle(coarse, levels - 1, sweep)
        sweep(r, x)
    return x


def _pcg(b, levels, its):
    """PCG on each grid of the leading axis: (x, |r|, |r0|)."""
    def dot(u, v):
        return (u * v).sum((-1, -2, -3), keepdim=True)
    x, r = torch.zeros_like(b), b.clone()
    norm0, p, rz = dot(r, r).sqrt(), None, None
    for _ in range(its):
        z = _vcycle(r, levels, _colour_sweep)
        old, rz = rz, dot(r, z)
        p = z if p is None else z + (rz / old) * p
        ap = _apply(p)
        alpha = rz / dot(p, ap)
        x += alpha * p
        r -= alpha * ap
    return x, dot(r, r).sqrt().reshape(-1), norm0.reshape(-1)


def _device_order(dims, where):
    """Natural row (grid by grid, x fastest) of each device row."""
    spot = torch.empty(8, dtype=torch.uint8, device=where)
    spot[torch.tensor(_SWEEP, device=where)] = torch.arange(8, dtype=torch.uint8, device=where)
    keys = []
    for nx, ny, nz in dims:
        c = [torch.arange(k, device=where) & 1 for k in (nz, ny, nx)]
        keys.append(spot[(4 * c[0][:, None, None] + 2 * c[1][:, None] + c[2]).reshape(-1)])
    return torch.sort(torch.cat(keys), stable=True)[1]


def exact(case, seed):
    kind, dims, s = case["kind"], _dims(case), case.get("s")
    b = _uniform(case, seed, 0, s)
    order = _device_order(dims, b.device)

    def natural(v):
        out = torch.empty_like(v)
        out[order] = v
        return out

    if kind in ("symgs", "mg"):
        r = natural(b).view(dims[0][::-1])
        if kind == "mg":
            x = _vcycle(r, case["levels"], _lex_sweep)
        else:
            x = natural(_uniform(case, seed, 1)).view(dims[0][::-1])
            _colour_sweep(r, x)
        return x.reshape(-1)[order]
    b = natural(b)
    got, at = [], 0
    for nx, ny, nz in dims:
        part = b[at:at + nx * ny * nz]
        at += nx * ny * nz
        grid = part.t() if s else part[None]
        got.append(_pcg(grid.reshape(-1, nz, ny, nx), case["levels"], case["its"]))
    if s:
        x = got[0][0].reshape(s, -1).t()
    else:
        x = torch.cat([g[0].reshape(-1) for g in got])
    one = kind in ("cg", "mixed")
    normr, normr0 = (torch.cat([g[k] for g in got]).cpu() for k in (1, 2))
    return dict(x=x[order], niters=None, normr=normr[0] if one else normr,
                normr0=normr0[0] if one else normr0)
