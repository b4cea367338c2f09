"""One FP64 RK stage of 1-D, 2-D and 3-D grids against the oracle with options
drawn at random: extents, stretched coordinates, boundary pairs, number of
components, viscosity and gravity on or off, resistivity in both forms,
Powell's sources, tiles or one line pass per axis.  Increments at 1e-11, states
and maxviscoef at 1e-12, as for the other random stages; an increment below
1e-4 of its state is measured by that (the state's own rounding is 1e-16)."""
import numpy as np
import pytest

from sac_amd import problems
from tests.helpers import make_oracle, mesh, per_var_errors, perturbed

pytestmark = pytest.mark.gpu

PAIRS = [("periodic", "periodic"), ("cont", "cont"), ("fixed", "fixed"), ("cont1", "grad1"),
         ("symm", "asymm"), ("fixed1", "cont"), ("contCD4", "symm0"), ("asymm", "fixed")]
LEFT = {"rho": 1.0, "p": 0.8, "v": [0.1, -0.2, 0.3], "b": [0.6, 0.5, -0.4]}
RIGHT = {"rho": 0.3, "p": 0.2, "v": [-0.1, 0.2, 0.0], "b": [0.6, 0.5, 0.4]}


def _draw(seed):
    rng = np.random.default_rng(90000 + seed)
    ndim = int(rng.integers(1, 4))
    if ndim == 3:
        # some with enough columns for the z work by columns
        nxyz = (tuple(int(x) for x in rng.integers(6, 40, size=3)) if seed % 3 else
                (int(rng.integers(90, 150)), int(rng.integers(120, 160)), int(rng.integers(62, 90))))
        prob = problems.stratified(n=nxyz[0], nxyz=nxyz, amp=3e-2)
    elif ndim == 2:
        prob = problems.riemann_patch(int(rng.integers(6, 70)), int(rng.integers(6, 70)),
                                      LEFT, RIGHT)
        if seed % 4 == 0:  # two components: the third's momentum and field go
            keep = [0, 1, 2, 4, 5, 6, 8, 9, 10, 11]
            prob.w, prob.ndir, prob.typeB = prob.w[keep].copy(), 2, prob.typeB[keep].copy()
    elif seed % 2:
        prob = problems.riemann_tube(int(rng.integers(6, 300)), LEFT, RIGHT)
    else:
        prob = problems.brio_wu(n=int(rng.integers(6, 300)))
    if ndim < 3:
        for k in range(prob.ndir):  # a background to work against
            prob.w[-prob.ndir + k][prob.mesh_slices()] = 0.1 * (k + 1)
        prob.w[2 * prob.ndir + 2][prob.mesh_slices()] = 0.7
        prob.w[2 * prob.ndir + 3][prob.mesh_slices()] = 0.2
    codes = []
    for d in range(ndim):
        codes += PAIRS[int(rng.integers(len(PAIRS)))]
        if rng.random() < 0.5:  # stretched along axis d
            prob.x[d] = prob.x[d] + 0.1 * np.sin(2.0 * prob.x[d] + d)
    prob.typeB[:, :] = np.array([problems.BC[c] for c in codes], dtype=np.int32)[None, :]
    for d in range(3):
        prob.eqpar[3 + d] = float(rng.normal()) if rng.random() < 0.6 else 0.0
    prob.eqpar[5] = float(rng.choice([1.0, 0.3, 0.0]))  # viscosity's switch, and g3
    prob.eqpar[1] = 1e-3 if prob.ndir > 1 and rng.random() < 0.4 else 0.0
    opt = {"divb": bool(rng.random() < 0.4), "compact": bool(rng.random() < 0.5),
           "tiles": bool(rng.random() < 0.8)}
    return prob, codes, opt


def _increments(prob, got, ref, w0, ne):
    """per variable: L2 of the difference of increments, relative to the
    increment's or, where that is larger, to 1e-4 of the state's"""
    out = []
    for v in range(ne):
        g, r, w = (mesh(prob, a[v]) for a in (got, ref, w0))
        size = max(np.linalg.norm(r - w), 1e-4 * np.linalg.norm(w), 1e-300)
        out.append(np.linalg.norm((g - w) - (r - w)) / size)
    return out


@pytest.mark.parametrize("seed", range(48))
def test_stage_matches_oracle(oracle_mod, seed):
    from sac_amd import device
    prob, codes, opt = _draw(seed)
    ne = 2 + 2 * prob.ndir
    o = make_oracle(prob, oracle_mod)
    o.set_divbfix(opt["divb"])
    o.set_resistive(opt["compact"])
    w0 = o.get_w()
    wct = perturbed(type(prob)(**{**prob.__dict__, "w": w0.copy()}), seed=seed, amp=1e-2).w
    wct = o.getboundary_on(wct)
    ref = o.advect1(1e-3, wct, w0)
    what = f"{prob.nx} ndir={prob.ndir} {codes} {opt} eqpar={prob.eqpar}"
    dev = device.Device(prob)
    try:
        dev.set_plane_tiles(opt["tiles"])
        dev.set_divbfix(opt["divb"])
        dev.set_resistive(opt["compact"])
        dev.upload(prob.w)
        dev.getboundary()
        dev.upload_slot(device.SLOT_S1, wct)
        dev.upload_slot(device.SLOT_S2, w0)
        dev.advect1(1e-3, device.SLOT_S1, device.SLOT_S2)
        got = dev.download_slot(device.SLOT_S2)
        mv = dev.maxviscoef
    finally:
        dev.close()
    inc = _increments(prob, got, ref, w0, ne)
    assert max(inc) <= 1e-11, f"{what}: increments {inc}"
    st = per_var_errors(prob, got, ref, ne)
    assert max(st) <= 1e-12, f"{what}: states {st}"
    assert mv == pytest.approx(o.maxviscoef, rel=1e-12), what
