"""Stages on 16 x 16 tiles (2-D grids in one launch): one RK4 step at extents
around the tile edges (tiles start at the first mesh cell along both axes;
test_tile_edges.py has the extents that end one along x), every boundary type,
with Powell's sources and resistivity, against the oracle in FP64 at 1e-12 per
variable and at FP32 resolution (1e-5, as in the other tests of the mixed
form), and against the schedule of one line pass per axis."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import assert_close_state, make_oracle, per_var_errors, perturbed

pytestmark = pytest.mark.gpu

LEFT = {"rho": 1.0, "p": 0.8, "v": [0.1, -0.2, 0.3], "b": [0.6, 0.5, -0.4]}
RIGHT = {"rho": 0.3, "p": 0.2, "v": [-0.1, 0.2, 0.0], "b": [0.6, 0.5, 0.4]}


def _patch(nx, ny, codes=None, eta=0.0):
    prob = perturbed(problems.riemann_patch(nx, ny, LEFT, RIGHT), seed=nx * 100 + ny, amp=1e-2)
    if codes:
        prob.typeB[:, :] = np.array([problems.BC[c] for c in codes], dtype=np.int32)[None, :]
    prob.eqpar[1] = eta
    return prob


def _step(device, oracle_mod, prob, precision="fp64", divb=False, tiles=True):
    dev = device.Device(prob, precision=precision)
    try:
        dev.set_plane_tiles(tiles)
        dev.set_divbfix(divb)
        dev.upload(prob.w)
        dev.getboundary()
        dt = dev.step(prob.courantpar)
        return dev.download(), dt, dev.maxviscoef
    finally:
        dev.close()


@pytest.mark.parametrize("nx", [6, 13, 14, 15, 30, 47])
@pytest.mark.parametrize("ny", [6, 15, 16, 17, 33])
def test_sizes(oracle_mod, nx, ny):
    from sac_amd import device
    prob = _patch(nx, ny)
    o = make_oracle(prob, oracle_mod)
    dt = o.step(prob.courantpar)
    w, got, mv = _step(device, oracle_mod, prob)
    assert abs(got - dt) <= 1e-13 * dt
    assert_close_state(prob, w, o.get_w(), 1e-12, 8, f"{nx}x{ny}")
    assert mv == pytest.approx(o.maxviscoef, rel=1e-10)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("codes", [("periodic", "periodic", "periodic", "periodic"),
                                   ("symm", "asymm", "contCD4", "fixed"),
                                   ("cont1", "grad1", "fixed1", "cont")])
@pytest.mark.parametrize("divb,eta", [(False, 0.0), (True, 0.0), (True, 1e-3)])
def test_options(oracle_mod, precision, tol, codes, divb, eta):
    from sac_amd import device
    prob = _patch(31, 18, codes, eta)
    o = make_oracle(prob, oracle_mod)
    o.set_divbfix(divb)
    o.step(prob.courantpar)
    w, _, _ = _step(device, oracle_mod, prob, precision, divb)
    assert_close_state(prob, w, o.get_w(), tol, 8, str(codes))
    line, _, _ = _step(device, oracle_mod, prob, precision, divb, tiles=False)
    assert max(per_var_errors(prob, w, line, 8)) <= tol
