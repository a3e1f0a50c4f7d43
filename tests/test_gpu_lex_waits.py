"""Reference-order sweeps whose waits give up are reported.  A limit of 0 polls
(tune "lex_polls") makes every wait that is not met at once give up; the
kernels still run to their end, with a wrong x."""
import os
import subprocess

import pytest

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host", "_bin", "wait_check")

pytestmark = pytest.mark.gpu


def limited(P, call):
    """The error of call() and of a check after it, under a limit of 0 polls."""
    from hpcg_amd._lib import HpcgxError
    P.tune("lex_polls", 0)
    try:
        call()
        P.check()
        return None
    except HpcgxError as e:
        return str(e)
    finally:
        P.tune("lex_polls", 1 << 22)


def test_lex_polls_reported():
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate(16, 16, 64, nlevels=2)
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    r = torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
    want = torch.zeros_like(r)
    P.mg(r, want, ordering="lexicographic")
    P.check()
    for call in (lambda: P.symgs(r, torch.zeros_like(r), ordering="lexicographic"),
                 lambda: P.mg(r, torch.zeros_like(r), ordering="lexicographic"),
                 lambda: P.cg(r, torch.zeros_like(r), max_iter=2, ordering="lexicographic")):
        assert "timed out" in (limited(P, call) or "")
        # reported once; later sweeps are right again
        P.check()
        z = torch.zeros_like(r)
        P.mg(r, z, ordering="lexicographic")
        P.check()
        assert torch.equal(z, want)
    P.close()


def test_lex_polls_reported_by_fleet_cg():
    import hpcg_amd
    import torch
    from hpcg_amd._lib import HpcgxError
    P = hpcg_amd.Problem.generate_fleet(((16, 16, 32), (8, 16, 24)), nlevels=1)
    b = torch.ones(P.nrow(0), dtype=torch.float64, device="cuda")
    for graph in (False, True):
        x = torch.zeros_like(b)
        P.tune("lex_polls", 0)
        with pytest.raises(HpcgxError, match="timed out"):
            P.cg_fleet(b, x, max_iter=3, ordering="lexicographic", graph=graph)
        P.tune("lex_polls", 1 << 22)
        P.check()
        outs = []
        for panels in (1, 0):
            P.tune("lex_panels", panels)
            x = torch.zeros_like(b)
            P.cg_fleet(b, x, max_iter=3, ordering="lexicographic", graph=graph)
            outs.append(x)
        P.tune("lex_panels", 1)
        assert torch.equal(*outs)
    P.close()


def test_lex_polls_reported_by_host_surface():
    """DeviceSYMGS and DeviceMG return the error (tests/host/wait_check.cpp)."""
    assert os.path.exists(CHECK), "wait_check not built (run __graft_entry__.build())"
    r = subprocess.run([CHECK], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0


def test_fleet_problems_do_not_wait_for_each_other():
    """One plane a problem: no panel couples to another, so no wait is left to
    give up, even under a limit of 0 polls."""
    import hpcg_amd
    import torch
    P = hpcg_amd.Problem.generate_fleet(((24, 16, 1), (8, 40, 1), (70, 9, 1)) * 8, nlevels=1)
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    r = torch.rand(P.nrow(0), generator=g, dtype=torch.float64, device="cuda") - 0.5
    x = torch.zeros_like(r)
    assert limited(P, lambda: P.symgs(r, x, ordering="lexicographic")) is None
    P.tune("lex_panels", 0)
    y = torch.zeros_like(r)
    P.symgs(r, y, ordering="lexicographic")
    assert torch.equal(x, y)
    P.close()
