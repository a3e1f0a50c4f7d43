"""The reference-order sweeps' copies make room for the problem's own state:
with about 2 GiB of the device left, the mixed-precision state of 256^3 (more
than 4 GiB) fits only once the copies (about 5 GiB) have gone."""
import pytest

pytestmark = pytest.mark.gpu


def test_copies_make_room():
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(256, 256, 256, nlevels=4)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    r = torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
    want, got = torch.empty_like(r), torch.empty_like(r)
    before = P.memory_use()
    P.mg(r, want, ordering="lexicographic")
    P.check()
    copies = P.memory_use() - before
    assert copies > 4 << 30
    free = torch.cuda.mem_get_info()[0]
    held = [torch.empty(free - (2 << 30), dtype=torch.uint8, device="cuda")]
    base = P.memory_use()
    P.prepare_mixed()
    torch.cuda.synchronize()
    assert P.memory_use() - base + copies > 4 << 30  # the state is there, the copies are not
    P.mg(r, got, ordering="lexicographic")  # by launches: no room for a copy
    P.check()
    assert torch.equal(got, want)
    held.clear()
    torch.cuda.empty_cache()
    P.close()
