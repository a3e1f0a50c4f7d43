"""What the reference-order sweeps' copy of a level costs, and where it is taken."""
import resource

import pytest

pytestmark = pytest.mark.gpu


def random_pair(n, seed=1):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return [torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
            for _ in range(2)]


def both(P, seed=1):
    """x after a sweep of the finest level by panels and by hyperplanes."""
    r, x = random_pair(P.nrow(0), seed)
    out = []
    for panels in (1, 0):
        P.tune("lex_panels", panels)
        y = x.clone()
        P.symgs(r, y, ordering="lexicographic")
        P.check()
        out.append(y)
    P.tune("lex_panels", 1)
    return out


def test_long_grid_host_memory():
    """Keys of the hyperplanes that a panel meets, not of all: on 16 x 16 x 4000 a
    table of panels by hyperplanes has 64 million entries, 8 bytes each."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(16, 16, 4000, nlevels=1)
    r, x = random_pair(P.nrow(0))
    torch.cuda.synchronize()
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss  # KiB
    P.symgs(r, x.clone(), ordering="lexicographic")
    P.check()
    grown = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before
    # steps and records of 4000 panels of 46 hyperplanes: 26 MB, and 2 MB of keys
    assert grown < 150 << 10, grown
    P.close()


@pytest.mark.parametrize("dims", [(1, 1, 500), (1, 7, 300), (3, 1, 400), (8, 8, 4000)])
def test_long_grids_same_bits(dims):
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(*dims, nlevels=1)
    a, b = both(P)
    assert torch.equal(a, b)
    P.close()


@pytest.mark.parametrize("dims", [(64, 48, 32), (130, 64, 20)])
def test_copy_bytes(dims):
    """No 32-bit columns (108 bytes a row) where the rows' offsets are regular."""
    import hpcg_amd
    P = hpcg_amd.Problem.generate(*dims, nlevels=1)
    n = P.nrow(0)
    r, x = random_pair(n)
    before = P.memory_use()
    P.symgs(r, x, ordering="lexicographic")
    P.check()
    # 28 values, x, r, three row ids; a 128-byte record per wavefront and step
    # (at most one step per two rows of these planes' shortest hyperplanes)
    grown = (P.memory_use() - before) / n
    assert 252 <= grown < 252 + 32, grown
    P.close()
