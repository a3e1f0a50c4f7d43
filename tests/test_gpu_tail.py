"""The V-cycle's smallest levels in one launch: the bits of the launches it
replaces, which other tests compare with the oracle.  Sizes: levels of one row
a colour and less than a tile; all tiles held in registers (at most 16);
colours of several tiles with a ragged last one; affine tiles and others; the
largest level (6000 rows) and one beyond it, whose coarser levels still run so."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [((2, 2, 2), 1), ((3, 3, 3), 1), ((8, 8, 8), 4), ((10, 10, 10), 1), ((9, 13, 7), 1),
         ((12, 20, 4), 3), ((16, 16, 16), 4), ((20, 20, 15), 1), ((40, 24, 56), 4),
         ((26, 22, 30), 2)]


@pytest.mark.parametrize("dims,levels", SIZES)
def test_tail_same_bits(dims, levels):
    import hpcg_amd
    import torch
    print("[case]", dims, levels, flush=True)
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    n = P.nrow(0)
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    b = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
    for c16 in (1, 0):
        P.tune("col16", c16)
        outs = []
        for tail in (1, 0):
            P.tune("tail", tail)
            z, z4 = torch.full_like(b, float("nan")), torch.full_like(b.float(), float("nan"))
            P.mg(b, z, ordering="multicolor")
            P.mg32(b.float(), z4, ordering="multicolor")
            got = [z, z4]
            for graph in (False, True):
                y = torch.zeros_like(b)
                P.cg(b, y, max_iter=3, tolerance=0.0, graph=graph)
                got.append(y)
            y = torch.zeros_like(b)
            P.cg_mixed(b, y, max_iter=3, tolerance=0.0)
            outs.append(got + [y])
        for k, (p, q) in enumerate(zip(*outs)):
            assert torch.equal(p, q) or (p.isnan().equal(q.isnan()) and k > 1), (c16, k)
    P.close()


def test_tail_streams():
    """Two streams at once: the launch keeps nothing outside its own x."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(16, 16, 16, nlevels=4)
    n = P.nrow(0)
    b = [torch.rand(n, dtype=torch.float64, device="cuda") for _ in range(2)]
    want = [torch.empty_like(v) for v in b]
    for v, w in zip(b, want):
        P.mg(v, w, ordering="multicolor")
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in b]
    got = [torch.empty_like(v) for v in b]
    for _ in range(10):
        for s, v, w in zip(streams, b, got):
            with torch.cuda.stream(s):
                P.mg(v, w, ordering="multicolor")
    torch.cuda.synchronize()
    for w, v in zip(want, got):
        assert torch.equal(w, v)
    P.close()


@pytest.mark.parametrize("s", [1, 2, 8, 64])
@pytest.mark.parametrize("dims,levels", [((3, 3, 3), 1), ((16, 16, 16), 4), ((24, 20, 28), 3)])
def test_tail_block_same_bits(dims, levels, s):
    """A workgroup per right-hand side: the bits of the block launches."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    B = torch.rand((P.nrow(0), s), generator=g, dtype=torch.float64, device="cuda") - 0.5
    outs = []
    for tail in (1, 0):
        P.tune("tail", tail)
        Z, X = torch.full_like(B.float(), float("nan")), torch.zeros_like(B)
        P.mg32_block(B.float(), Z, ordering="multicolor")
        P.cg_block_mixed(B, X, max_iter=3, recompute=2)
        outs.append((Z, X))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    P.close()
