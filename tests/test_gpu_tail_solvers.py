"""The one-launch levels inside the solvers: where the finest level runs so it
also leaves the r.z partials of the last sweep, in captured iterations too.  The
same bits as the launches, of x and of the residual norms, all finite.

Sizes: every level in the launch, with narrow column ids on the finest (4096
rows and more: without them no partials are left); colours of whole tiles,
colours with a ragged last tile, and the largest level; and a finest level
beyond it."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [((16, 16, 16), 4), ((20, 12, 24), 2), ((20, 20, 15), 1), ((18, 20, 16), 2),
         ((40, 24, 56), 4)]


@pytest.mark.parametrize("c16", [1, 0])
@pytest.mark.parametrize("dims,levels", SIZES)
def test_tail_solvers_same_bits(dims, levels, c16):
    import hpcg_amd
    import torch
    print("[case]", dims, levels, c16, flush=True)
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    g = torch.Generator(device="cuda")
    g.manual_seed(23)
    b = torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
    P.tune("col16", c16)
    outs = []
    for tail in (1, 0):
        P.tune("tail", tail)
        got = []
        for solve in (lambda x: P.cg(b, x, max_iter=4),
                      lambda x: P.cg(b, x, max_iter=4, graph=True),
                      lambda x: P.cg_mixed(b, x, max_iter=4)):
            x = torch.zeros_like(b)
            res = solve(x)
            assert x.isfinite().all() and 0.0 < res["normr"] < res["normr0"]
            got.append((x, res["normr"], res["normr0"]))
        outs.append(got)
    for k, (p, q) in enumerate(zip(*outs)):
        assert torch.equal(p[0], q[0]) and p[1:] == q[1:], k
    P.close()


def test_tail_fleet_same_bits():
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate_fleet(((8, 16, 16), (16, 8, 8), (8, 8, 24)), nlevels=2)
    g = torch.Generator(device="cuda")
    g.manual_seed(29)
    b = torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
    for graph in (False, True):
        outs = []
        for tail in (1, 0):
            P.tune("tail", tail)
            x = torch.zeros_like(b)
            res = P.cg_fleet(b, x, max_iter=4, graph=graph)
            assert x.isfinite().all()
            outs.append((x, res["normr"]))
        assert torch.equal(outs[0][0], outs[1][0]) and outs[0][1] == outs[1][1]
    P.close()
