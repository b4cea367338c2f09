"""One RK4 step of 1-D grids at sizes around the tiles of the one-launch
stage (64 cells up to 32768 cells; test_stage1_long.py has the grids on tiles
of 256), against the oracle: a step's rounding differences stay at a few 1e-16
per variable, the bar is 1e-12."""
import pytest

from sac_amd import problems
from tests.helpers import assert_close_state, oracle_run, perturbed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [6, 63, 64, 65, 4096, 4097, 4353])
@pytest.mark.parametrize("ndir", [2, 3])
def test_one_step_matches_oracle(oracle_mod, n, ndir):
    from sac_amd import device
    if ndir == 2:
        prob = problems.brio_wu(n=n)
    else:
        prob = problems.riemann_tube(n, {"rho": 1.0, "p": 0.8, "v": [0.1, -0.2, 0.3],
                                         "b": [0.6, 0.5, -0.4]},
                                     {"rho": 0.3, "p": 0.2, "v": [-0.1, 0.2, 0.0],
                                      "b": [0.6, -0.5, 0.4]})
    perturbed(prob, seed=n, amp=1e-2)
    ref, dts, _ = oracle_run(prob, oracle_mod, 1)
    w, got = device.run(prob, steps=1)
    assert abs(got[0] - dts[0]) <= 1e-13 * dts[0]
    assert_close_state(prob, w, ref, 1e-12, 2 + 2 * ndir, f"n={n}")


def test_maxviscoef_is_taken_once():
    """getdt_special takes maxviscoef: it reads 0 (and limits no dt) until the
    next stage, and a value set by hand counts as one of a stage."""
    from sac_amd import device
    prob = perturbed(problems.brio_wu(n=100), seed=3, amp=1e-2)
    dev = device.Device(prob)
    try:
        dev.upload(prob.w)
        dev.getboundary()
        assert dev.maxviscoef == 0.0
        dev.advance(1e-5)
        mv = dev.maxviscoef
        assert mv > 0.0
        dx2 = float(dev.dx[2:-2].min()) ** 2
        assert dev.getdt_special(1.0) == min(1.0, 0.25 / (mv / dx2))
        assert dev.maxviscoef == 0.0 and dev.getdt_special(1.0) == 1.0
        dev.maxviscoef = mv
        assert dev.maxviscoef == mv
        # a stage keeps the larger of the two
        dev.advance(1e-5)
        assert dev.maxviscoef >= mv
        dev.getdt_special(1.0)
        dev.copy_slot(device.SLOT_S1, device.SLOT_W)
        dev.advect1(1e-6, device.SLOT_S1, device.SLOT_W)
        assert 0.0 < dev.maxviscoef
    finally:
        dev.close()
