"""The one-launch levels of problems of different sizes, used by a thread each:
their LDS needs differ (8 to 96 KiB), and no thread's launch depends on
another's."""
import threading

import pytest

pytestmark = pytest.mark.gpu

SIZES = [((8, 8, 8), 2), ((16, 16, 16), 4), ((20, 20, 15), 1), ((10, 10, 10), 1)]


def test_tail_threads():
    import hpcg_amd
    import torch
    probs = [hpcg_amd.Problem.generate(*d, nlevels=l) for d, l in SIZES]
    rs = [torch.linspace(-1.0, 1.0, P.nrow(0), dtype=torch.float64, device="cuda") for P in probs]
    want, want32 = [], []
    for P, r in zip(probs, rs):
        P.prepare_mixed()
        P.tune("tail", 0)
        z, z32 = torch.empty_like(r), torch.empty_like(r.float())
        P.mg(r, z, ordering="multicolor")
        P.mg32(r.float(), z32, ordering="multicolor")
        P.tune("tail", 1)
        want.append(z)
        want32.append(z32)
    torch.cuda.synchronize()
    fails = []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(100):
                    z, z32 = torch.empty_like(rs[k]), torch.empty_like(want32[k])
                    probs[k].mg(rs[k], z, ordering="multicolor")
                    probs[k].mg32(rs[k].float(), z32, ordering="multicolor")
                    if not (torch.equal(z, want[k]) and torch.equal(z32, want32[k])):
                        fails.append(k)
        except Exception as e:  # (reported by the test's own thread)
            fails.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(SIZES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not fails, fails
    for P in probs:
        P.close()
