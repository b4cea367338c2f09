"""Line passes of small 3-D grids march segments of one or two 16-point chunks
(10 and 26 cells after the halo): one RK4 step at line lengths around the
ends of a segment, along z alone (the other axes on tiles) and along y and z
(one line pass per axis), against the oracle in FP64 at 1e-12 per variable,
with the maximal viscosity coefficient of the step."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import assert_close_state, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nxyz", [(9, 8, 6), (9, 10, 10), (18, 11, 11), (7, 20, 21), (10, 26, 27),
                                  (33, 27, 53)])
@pytest.mark.parametrize("tiles", [True, False])
def test_lengths(oracle_mod, nxyz, tiles):
    from sac_amd import device
    prob = problems.stratified(n=nxyz[0], nxyz=nxyz, amp=3e-2)
    prob.typeB[:, 4:] = np.int32(problems.BC["periodic"])
    o = make_oracle(prob, oracle_mod)
    dt = o.step(prob.courantpar)
    dev = device.Device(prob)
    try:
        dev.set_plane_tiles(tiles)
        dev.upload(prob.w)
        dev.getboundary()
        got = dev.step(prob.courantpar)
        assert abs(got - dt) <= 1e-13 * dt
        assert_close_state(prob, dev.download(), o.get_w(), 1e-12, 8, str(nxyz))
        assert dev.maxviscoef == pytest.approx(o.maxviscoef, rel=1e-10)
    finally:
        dev.close()
