"""One RK4 step of long 1-D grids, around the cell count at which the one-launch
stage changes from tiles of 64 cells to tiles of 256 (32768), and with a last
tile of one cell, against the oracle: a step's rounding differences stay at a
few 1e-16 per variable, the bar is 1e-12."""
import pytest

from sac_amd import problems
from tests.helpers import assert_close_state, oracle_run, perturbed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32767, 32768, 32769, 33024, 33025])
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
