"""The z work of 3-D grids by columns (grids with many columns): one RK4 step
at sizes with ragged rows and blocks and with segments of every kind (one
short one, full ones, a last one of one cell), open and periodic in z, with
Powell's sources, against the oracle in FP64 at 1e-12 per variable and at FP32
resolution (1e-5, as in the other tests of the mixed form), and against the
schedule of one line pass per axis."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import assert_close_state, make_oracle, per_var_errors

pytestmark = pytest.mark.gpu


def _step(device, prob, precision, divb, tiles):
    dev = device.Device(prob, precision=precision)
    try:
        dev.set_plane_tiles(tiles)
        dev.set_divbfix(divb)
        dev.upload(prob.w)
        dev.getboundary()
        dev.step(prob.courantpar)
        return dev.download(), dev.maxviscoef
    finally:
        dev.close()


@pytest.mark.parametrize("nxyz,zbc,divb", [
    ((300, 257, 7), "cont", False),      # one segment shorter than 16 cells
    ((200, 130, 33), "periodic", True),  # 16 + 16 + 1 cells
    ((61, 75, 203), "fixed", False),     # many segments of few columns
    ((391, 340, 40), "cont", True),      # 32 + 8 cells
])
def test_step_matches_oracle(oracle_mod, nxyz, zbc, divb):
    from sac_amd import device
    prob = problems.stratified(n=nxyz[0], nxyz=nxyz, amp=3e-2, noise=1e-3)
    prob.typeB[:, 4:] = np.int32(problems.BC[zbc])
    o = make_oracle(prob, oracle_mod)
    o.set_divbfix(divb)
    o.step(prob.courantpar)
    ref = o.get_w()
    for precision, tol in (("fp64", 1e-12), ("mixed", 1e-5)):
        w, mv = _step(device, prob, precision, divb, True)
        assert_close_state(prob, w, ref, tol, 8, f"{nxyz} {precision}")
        line, mv_line = _step(device, prob, precision, divb, False)
        assert max(per_var_errors(prob, w, line, 8)) <= tol
        if precision == "fp64":
            assert mv == pytest.approx(o.maxviscoef, rel=1e-10)
            assert mv == pytest.approx(mv_line, rel=1e-10)
