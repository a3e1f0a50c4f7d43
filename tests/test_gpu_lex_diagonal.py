"""A replaced diagonal reaches the reference-order sweeps' copy of the matrix
whatever the diagonal was when the copy was built: the same bits as one launch
per hyperplane, which reads the matrix itself."""
import pytest

pytestmark = pytest.mark.gpu


def sweeps(P, level=0, seed=3):
    """x after a sweep by panels and by hyperplanes."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r, x = (torch.rand(P.nrow(level), generator=g, dtype=torch.float64, device="cuda") - 0.5
            for _ in range(2))
    out = []
    for panels in (1, 0):
        P.tune("lex_panels", panels)
        y = x.clone()
        P.symgs(r, y, level=level, ordering="lexicographic")
        P.check()
        out.append(y)
    P.tune("lex_panels", 1)
    return out


@pytest.mark.parametrize("every", [1, 7])
@pytest.mark.parametrize("dims", [(3, 3, 3), (20, 18, 11), (64, 48, 8)])
def test_diagonal_zero_when_copied(dims, every):
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(*dims, nlevels=1)
    d = P.copy_diagonal()
    z = d.clone()
    z[::every] = 0.0
    P.replace_diagonal(z)
    sweeps(P)  # builds the copy; its x holds infinities
    P.replace_diagonal(d * 1.25)
    a, b = sweeps(P)
    assert a.isfinite().all() and torch.equal(a, b)
    P.close()


def test_captured_replacements():
    """A replacement captured before the copy exists, and one captured after,
    each replayed with new values between sweeps; and one by the CG's own graph."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(24, 40, 16, nlevels=2)
    d = [P.copy_diagonal(l) for l in range(2)]
    new = [v.clone() for v in d]
    graphs = []
    for when in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for l in range(2):
                P.replace_diagonal(new[l], l)
        graphs.append(graph)
        for k in range(3):
            for graph in graphs:
                for l in range(2):
                    new[l].copy_(d[l] * (1.0 + 0.1 * (3 * when + k + 1)))
                graph.replay()
                for l in range(2):
                    a, b = sweeps(P, l, seed=k)
                    assert a.isfinite().all() and torch.equal(a, b), (when, k, l)
    outs = []
    r = torch.ones(P.nrow(0), dtype=torch.float64, device="cuda")
    for panels in (1, 0):
        P.tune("lex_panels", panels)
        for l in range(2):
            P.replace_diagonal(d[l], l)
        x = [torch.zeros_like(r) for _ in range(2)]
        P.cg(r, x[0], max_iter=3, ordering="lexicographic", graph=True)
        for l in range(2):
            P.replace_diagonal(d[l] * 1.5, l)
        P.cg(r, x[1], max_iter=3, ordering="lexicographic", graph=True)
        outs.append(x)
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert not torch.equal(outs[0][0], outs[0][1])
    P.close()
