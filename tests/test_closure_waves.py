"""Inference of the learned closure leaves the network out in wavefronts none
of whose 64 faces use it and takes the axes of a stage in one launch.  Which
faces share a wavefront follows from where the structure lies on the grid, and
the result must not: a localised pulse (flat elsewhere, twenty cells and more
from every edge, whose layers the scheme treats in its own way), moved by a
few cells, gives the moved result.  Extents are powers of two (the coordinates
are exact), so no face changes its side of the sensor's thresholds; 1e-12 per
variable, and the network must have mattered."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import per_var_errors

pytestmark = pytest.mark.gpu

STATE = {"rho": 1.0, "p": 0.8, "v": [0.0, 0.0, 0.0], "b": [0.6, 0.5, -0.4]}


def _problem(nx, shift):
    if len(nx) == 3:
        prob = problems.stratified(n=nx[0], nxyz=nx, amp=0.0, noise=0.0)
    elif len(nx) == 2:
        prob = problems.riemann_patch(nx[0], nx[1], STATE, STATE)
    else:
        prob = problems.riemann_tube(nx[0], dict(STATE), dict(STATE))
    prob.typeB[:, 2 * (len(nx) == 3):] = np.int32(problems.BC["periodic"])
    ms = (Ellipsis,) + prob.mesh_slices()
    mesh = prob.w[ms].copy()
    # array axes are (z, y, x); the pulse sits in the middle of each
    grids = np.meshgrid(*[np.arange(n) - n / 2 for n in mesh.shape[1:]], indexing="ij")
    pulse = 0.05 * np.exp(-sum(a * a for a in grids) / 8.0)
    rho = mesh[0] + (mesh[-1 - prob.ndir] if len(nx) == 3 else 0.0)
    mesh[1] += rho * pulse
    mesh[1 + prob.ndir] += 0.1 * pulse
    prob.w[ms] = _moved(mesh, shift, len(nx))
    return prob


def _moved(mesh, shift, ndim):
    """mesh (variables, z, y, x) moved along its periodic axes: y and z of a
    3-D grid, all of the others."""
    for k, n in enumerate(shift):
        axis = k + (ndim == 3)
        mesh = np.roll(mesh, n, axis=mesh.ndim - 1 - axis)
    return mesh


def _run(prob, learned):
    from sac_amd import closure, device
    dev = device.Device(prob)
    try:
        dev.upload(prob.w)
        dev.getboundary()
        if learned:
            cl = closure.Closure(dev, capacity=0, max_blocks=8, seed=5)
            cl.enable(True, 0.5)
        for _ in range(2):
            dev.advance(1e-3)
        return dev.download()
    finally:
        dev.close()


@pytest.mark.parametrize("nx,shift", [((256,), (37,)), ((128, 64), (9, 3)), ((64, 128), (1, 13)),
                                      ((8, 64, 64), (5, 7)), ((16, 64, 64), (1, 9))])
def test_result_moves_with_the_structure(nx, shift):
    base, moved = _problem(nx, [0] * len(shift)), _problem(nx, shift)
    a, b = _run(base, True), _run(moved, True)
    plain = _run(base, False)
    ms = (Ellipsis,) + base.mesh_slices()
    ref = a.copy()
    ref[ms] = _moved(a[ms], shift, len(nx))
    got = a.copy()
    got[ms] = b[ms]
    assert max(per_var_errors(base, got, ref, 2 + 2 * base.ndir)) <= 1e-12
    assert np.abs(a[ms] - plain[ms]).max() > 1e-9
