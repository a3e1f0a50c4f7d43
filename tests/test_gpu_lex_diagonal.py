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
