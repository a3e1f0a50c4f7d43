"""Narrow column ids on levels whose colours start anywhere (tiles counted from
each colour's first row) and the colour steps with all of a row's loads in
flight: the bits of the 32-bit column ids, which other tests compare with the
oracle.  Sizes: fewer rows than a tile; colours shorter than a tile and of no
multiple of it; tiles over several grid lines and planes; one tile per line;
steps on both sides of the largest all-in-flight step (6 * 2^20 rows)."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [((3, 5, 4), 1), ((9, 7, 5), 1), ((17, 13, 11), 1), ((26, 22, 30), 2), ((40, 24, 56), 4),
         ((128, 6, 10), 1), ((151, 33, 20), 1), ((258, 30, 14), 2), ((400, 368, 344), 1)]


@pytest.mark.parametrize("dims,levels", SIZES)
def test_tiles_same_bits(dims, levels):
    import hpcg_amd
    import torch
    print("[case]", dims, levels, flush=True)
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    big = P.nrow(0) > 1 << 24
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    outs = []
    for c16 in (1, 0):
        P.tune("col16", c16)
        g.manual_seed(5)
        got = []
        for l in range(levels):
            n = P.nrow(l)
            r, x = (torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
                    for _ in range(2))
            y = torch.empty_like(x)
            P.spmv(x, y, level=l)
            P.symgs(r, x, level=l, ordering="multicolor")
            got += [y, x]
            x4 = x.float()
            P.symgs32(r.float(), x4, level=l, ordering="multicolor")
            got.append(x4)
        z = torch.empty_like(got[1])
        b = torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
        P.mg(b, z, ordering="multicolor")
        z4 = torch.empty_like(z.float())
        P.mg32(b.float(), z4, ordering="multicolor")
        got += [z, z4]
        if not big:
            B = torch.rand((P.nrow(0), 8), generator=g, dtype=torch.float64, device="cuda")
            Y, Z = torch.empty_like(B), torch.empty_like(B.float())
            P.spmv_block(B, Y)
            P.mg32_block(B.float(), Z, ordering="multicolor")
            got += [Y, Z]
        outs.append(got)
    for k, (a, b) in enumerate(zip(*outs)):
        assert torch.equal(a, b), k
    P.close()


@pytest.mark.parametrize("s", [4, 8, 16])
@pytest.mark.parametrize("dims,levels", [((3, 5, 4), 1), ((17, 13, 11), 1), ((40, 24, 56), 4),
                                         ((130, 66, 62), 2)])
def test_block_tiles_same_bits(dims, levels, s):
    """Row pointers from the tile's record and values two to a word, workgroups
    in windows of 64 (whole windows and a partial last one): the bits of the
    packed words and of the 32-bit ids."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    B = torch.rand((P.nrow(0), s), generator=g, dtype=torch.float64, device="cuda") - 0.5
    outs = []
    for knobs in ({"x_pairs": 1, "col16": 1}, {"x_pairs": 0, "col16": 1}, {"col16": 0}):
        for k, v in knobs.items():
            P.tune(k, v)
        Y, Z = torch.empty_like(B), torch.empty_like(B.float())
        P.spmv_block(B, Y)
        P.mg32_block(B.float(), Z, ordering="multicolor")
        outs.append((Y, Z))
    for got in outs[1:]:
        assert torch.equal(got[0], outs[0][0]) and torch.equal(got[1], outs[0][1])
    P.close()


@pytest.mark.parametrize("dims,levels", SIZES)
def test_turn_same_bits(dims, levels):
    """The turn of a symmetric sweep in one launch: the bits of the two colour
    steps, from any x and from x = 0, with narrow and 32-bit ids (where the
    FP64 steps stay apart), and r.z as a sum over the same partials."""
    import hpcg_amd
    import torch
    print("[case]", dims, levels, flush=True)
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    n = P.nrow(0)
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    b, x0 = (torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
             for _ in range(2))
    s = 8 if n < 1 << 20 else 0
    B = torch.rand((n, 10), generator=g, dtype=torch.float32, device="cuda") - 0.5
    for c16 in (1, 0):
        P.tune("col16", c16)
        outs = []
        for turn in (1, 0):
            P.tune("turn", turn)
            x, z, z4, x4 = x0.clone(), torch.empty_like(b), torch.empty_like(B[:, 0]), x0.float()
            P.symgs(b, x, ordering="multicolor")
            P.mg(b, z, ordering="multicolor")
            P.symgs32(b.float(), x4, ordering="multicolor")
            P.mg32(b.float(), z4, ordering="multicolor")
            got = [x, z, x4, z4]
            for lo, hi in ((0, 8), (8, 10)) if s else ():
                R = B[:, lo:hi].contiguous()
                Z = torch.empty_like(R)
                P.mg32_block(R, Z, ordering="multicolor")
                got.append(Z)
            for solve in (P.cg, P.cg_mixed):
                y = torch.zeros_like(b)
                got.append(torch.tensor(float(solve(b, y, max_iter=4, tolerance=0.0)["normr"])))
                got.append(y)
            outs.append(got)
        for k, (p, q) in enumerate(zip(*outs)):
            assert torch.equal(p, q), (c16, k)
    P.close()


@pytest.mark.parametrize("dims,levels", [((17, 13, 11), 1), ((130, 66, 62), 2), ((258, 30, 14), 2),
                                         ((128, 64, 64), 3)])
def test_half_spmv_same_bits(dims, levels):
    """The mixed solve's A p and residual from FP16 value pairs, on affine tiles
    with every load in flight (with and without shared x windows) and on others:
    the bits of the packed words."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(*dims, nlevels=levels)
    g = torch.Generator(device="cuda")
    g.manual_seed(13)
    b, x0 = (torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
             for _ in range(2))
    outs = []
    for hp in (1, 0):
        P.tune("hc_pairs", hp)
        x = x0.clone()
        r = P.cg_mixed(b, x, max_iter=5, tolerance=0.0, recompute=2)
        outs.append((x, r["normr"]))
    assert torch.equal(outs[0][0], outs[1][0]) and outs[0][1] == outs[1][1]
    P.close()
