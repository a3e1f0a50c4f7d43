"""The autotuner keeps the defaults of knobs that no launch of the problem
depends on, whatever the noise of its timings: "gs_waves" and "x_pairs" on
colour steps of at most 6 * 2^20 rows of a matrix that is not streamed."""
import pytest

pytestmark = pytest.mark.gpu


def test_autotune_keeps_idle_knobs():
    import hpcg_amd
    P = hpcg_amd.Problem.generate(24, 16, 16, nlevels=2)
    for _ in range(6):
        rep = P.autotune(iterations=1)
        assert "chosen gs_waves=1" in rep and "chosen x_pairs=3" in rep, rep
    P.close()
