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


@pytest.mark.parametrize("thread", [False, True])
def test_first_sweep_beside_a_capture(thread):
    """The first sweep allocates its copy; a capture on another stream, by this
    thread or another, stays valid and the copy is built."""
    import threading

    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(24, 16, 12, nlevels=1)
    n = P.nrow(0)
    r, x = random_pair(n)
    y = torch.zeros_like(x)
    side = torch.cuda.Stream()
    before = P.memory_use()
    z, fails = x.clone(), []

    def sweep():
        try:
            with torch.cuda.stream(side):
                P.symgs(r, z, ordering="lexicographic")
        except Exception as e:  # (reported by the test's own thread)
            fails.append(e)

    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y.copy_(x)
        if thread:
            t = threading.Thread(target=sweep)
            t.start()
            t.join()
        else:
            sweep()
    graph.replay()
    torch.cuda.synchronize()
    assert not fails, fails
    P.check()
    assert torch.equal(x, y)
    assert P.memory_use() - before >= 252 * n
    P.tune("lex_panels", 0)
    w = x.clone()
    P.symgs(r, w, ordering="lexicographic")
    assert torch.equal(z, w)
    P.close()


@pytest.mark.parametrize("dims,panels", [((512, 512, 1), True), ((4500, 4500, 1), False),
                                         ((1, 1, 2), False), ((1, 1, 3), True)])
def test_rule_for_panels(dims, panels):
    """A plane so wide that one workgroup takes longer over a hyperplane than a
    launch, and a level of two hyperplanes, keep one launch per hyperplane."""
    import hpcg_amd
    P = hpcg_amd.Problem.generate(*dims, nlevels=1)
    r, x = random_pair(P.nrow(0))
    before = P.memory_use()
    P.symgs(r, x, ordering="lexicographic")
    P.check()
    assert (P.memory_use() > before) == panels
    P.close()
