"""Mixed precision in other units of length: without gravity the equations
have no length of their own, so cell widths and dt multiplied by a power of two
multiply every rate by its inverse and leave each step's result as it is, bit
for bit, as long as no intermediate value leaves FP32's range.  At 2^80 the
widths are about 1e22 to 1e23 (centimetres in a galaxy), at 2^-80 about 1e-26:
1/dx is far inside FP32's range, 1/dx^2 is not."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import perturbed

pytestmark = pytest.mark.gpu

LEFT = {"rho": 1.0, "p": 0.8, "v": [0.1, -0.2, 0.3], "b": [0.6, 0.5, -0.4]}
RIGHT = {"rho": 0.3, "p": 0.2, "v": [-0.1, 0.2, 0.0], "b": [0.6, 0.5, 0.4]}


def _prob(n):
    if len(n) == 1:
        return perturbed(problems.riemann_tube(n[0], LEFT, RIGHT), seed=1, amp=1e-2)
    patch = problems.riemann_patch(n[0], n[1], LEFT, RIGHT)
    if len(n) == 2:
        return perturbed(patch, seed=2, amp=1e-2)
    # a patch's states in a box: the same planes along z
    prob = problems.stratified(n=n[0], nxyz=n)
    prob.w = np.repeat(patch.w, n[2] + 4, axis=1)
    prob.eqpar[3:6] = [0.0, 0.0, 1e-60]  # the last switches viscosity on; as a gravity it is nothing
    prob.typeB[:, :] = problems.BC["cont"]
    return perturbed(prob, seed=3, amp=1e-2)


def _steps(device, prob, scale, divb, tiles):
    dev = device.Device(prob, precision="mixed", dx=device.grid_dx(prob) * scale)
    try:
        dev.set_plane_tiles(tiles)
        dev.set_divbfix(divb)
        dev.upload(prob.w)
        dev.getboundary()
        dt = 0.05 * float(device.grid_dx(prob).min()) * scale
        for _ in range(2):
            dev.advance(dt)
        return dev.download(), dev.maxviscoef / scale
    finally:
        dev.close()


@pytest.mark.parametrize("n,tiles", [((70,), True), ((37, 29), True), ((37, 29), False),
                                     ((20, 18, 22), True), ((20, 18, 22), False),
                                     ((200, 130, 33), True)])  # z by columns
@pytest.mark.parametrize("power", [80, -80])
@pytest.mark.parametrize("divb", [False, True])
def test_mixed_steps_do_not_depend_on_the_unit(n, tiles, power, divb):
    from sac_amd import device
    prob = _prob(n)
    w, mv = _steps(device, prob, 1.0, divb, tiles)
    assert np.isfinite(w).all() and mv > 0.0
    got, gmv = _steps(device, prob, 2.0 ** power, divb, tiles)
    np.testing.assert_array_equal(got, w)
    assert gmv == mv
