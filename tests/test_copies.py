"""Uploads, downloads and saves: a state comes back as it went up, at sizes
of one small buffer, one chunk and several (4 MB), with rows that chunks cut
(a chunk of 2^19 FP64 elements is no multiple of these row lengths), in both
storage precisions (FP32: rounded once)."""
import numpy as np
import pytest

from sac_amd import problems

pytestmark = pytest.mark.gpu


def _prob(n):
    if len(n) == 1:
        prob = problems.riemann_tube(n[0], {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]},
                                     {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]})
    elif len(n) == 2:
        prob = problems.riemann_patch(*n, {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]},
                                      {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]})
    else:
        prob = problems.stratified(n=n[0], nxyz=n)
    rng = np.random.default_rng(sum(n))
    prob.w = prob.w + rng.standard_normal(prob.w.shape)
    prob.w[8:] = np.abs(prob.w[8:]) + 1.0
    return prob


@pytest.mark.parametrize("n", [(6,), (800,), (5039,), (5041,), (300001,), (61, 47), (255, 257),
                               (6, 6, 6), (31, 27, 35), (70, 61, 64)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_round_trip(n, precision):
    from sac_amd import device
    prob = _prob(n)
    want = prob.w.copy()
    if precision == "mixed":
        want[:8] = want[:8].astype(np.float32).astype(np.float64)
    dev = device.Device(prob, precision=precision)
    try:
        dev.upload(prob.w)
        np.testing.assert_array_equal(dev.download(), want)
        dev.save_begin()
        np.testing.assert_array_equal(dev.save_end(), want)
        other = prob.w[::-1].copy()
        dev.upload_slot(device.SLOT_S2, other)
        got = dev.download_slot(device.SLOT_S2)
        want[:8] = other[:8].astype(np.float32) if precision == "mixed" else other[:8]
        np.testing.assert_array_equal(got, want)
    finally:
        dev.close()


def test_ensemble_download():
    """Members of uneven sizes, one larger than a buffer; the evolving fields'
    mesh cells and the background's are those given."""
    from sac_amd import batch
    probs = [problems.riemann_patch(nx, ny, {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]},
                                    {"rho": 0.5, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]})
             for nx, ny in ((6, 6), (33, 17), (220, 230), (16, 64), (7, 150))]
    rng = np.random.default_rng(7)
    for p in probs:
        p.w[:8] += 1e-3 * rng.standard_normal(p.w[:8].shape)
    ens = batch.Ensemble(probs, tmax=1.0)
    try:
        for got, p in zip(ens.download(), probs):
            ms = (slice(None),) + p.mesh_slices()
            np.testing.assert_array_equal(got[ms], p.w[ms])
    finally:
        ens.close()
