"""Stages on 16 x 16 tiles at the x extents that fill a tile, end one cell into
the next and end one cell short (tiles start at the first mesh cell along both
axes), and z work by columns in FP32 storage at the fewest blocks that take it
(256): one RK4 step against the oracle, in FP64 at 1e-12 per variable and at
FP32 resolution (1e-5, as in the other tests of the mixed form)."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import assert_close_state, make_oracle, perturbed

pytestmark = pytest.mark.gpu

LEFT = {"rho": 1.0, "p": 0.8, "v": [0.1, -0.2, 0.3], "b": [0.6, 0.5, -0.4]}
RIGHT = {"rho": 0.3, "p": 0.2, "v": [-0.1, 0.2, 0.0], "b": [0.6, 0.5, 0.4]}


def _check(oracle_mod, prob, precisions):
    from sac_amd import device
    o = make_oracle(prob, oracle_mod)
    dt = o.step(prob.courantpar)
    ref = o.get_w()
    for precision, tol in precisions:
        dev = device.Device(prob, precision=precision)
        try:
            dev.upload(prob.w)
            dev.getboundary()
            got = dev.step(prob.courantpar)
            assert_close_state(prob, dev.download(), ref, tol, 8, f"{prob.nx} {precision}")
            if precision == "fp64":
                assert abs(got - dt) <= 1e-13 * dt
                assert dev.maxviscoef == pytest.approx(o.maxviscoef, rel=1e-10)
        finally:
            dev.close()


@pytest.mark.parametrize("nx", [15, 16, 17, 31, 32, 33, 48, 49])
@pytest.mark.parametrize("ny", [16, 17])
@pytest.mark.parametrize("xbc", ["cont", "periodic"])
def test_tile_ends_along_x(oracle_mod, nx, ny, xbc):
    prob = perturbed(problems.riemann_patch(nx, ny, LEFT, RIGHT), seed=nx * 100 + ny, amp=1e-2)
    prob.typeB[:, :2] = np.int32(problems.BC[xbc])
    _check(oracle_mod, prob, (("fp64", 1e-12), ("mixed", 1e-5)))


@pytest.mark.parametrize("nxyz", [(64, 64, 256),    # 16 blocks of columns, 16 segments: 256
                                  (64, 64, 255),    # the same, the last segment one cell short
                                  (65, 64, 256)])   # one column more: 17 blocks of columns
def test_fewest_columns_in_fp32(oracle_mod, nxyz):
    prob = problems.stratified(n=nxyz[0], nxyz=nxyz, amp=3e-2, noise=1e-3)
    _check(oracle_mod, prob, (("mixed", 1e-5),))
