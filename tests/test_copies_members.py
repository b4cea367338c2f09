"""Ensemble downloads whose members are larger than a buffer (4 MB) and whose
fields are cut by the chunks: the evolving fields' mesh cells and the
background's are those given, bit for bit."""
import numpy as np
import pytest

from sac_amd import problems

pytestmark = pytest.mark.gpu

SIDE = {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]}


@pytest.mark.parametrize("sizes", [
    [(n,) for n in (60001, 6, 300001, 800, 7, 40329, 40330)],  # 40330: 13 fields of 40334 in 4 MB less a few
    [(6, 6), (700, 611), (33, 17), (150, 260), (7, 150)],
])
def test_members_come_back(sizes):
    from sac_amd import batch
    make = problems.riemann_tube if len(sizes[0]) == 1 else problems.riemann_patch
    probs = [make(*n, SIDE, SIDE) for n in sizes]
    rng = np.random.default_rng(11)
    for p in probs:
        p.w[:8] += 1e-3 * rng.standard_normal(p.w[:8].shape)
        p.w[8:] = 1e-3 * rng.random(p.w[8:].shape)
    ens = batch.Ensemble(probs, tmax=1.0)
    try:
        for got, p in zip(ens.download(), probs):
            ms = (slice(None),) + p.mesh_slices()
            np.testing.assert_array_equal(got[ms], p.w[ms])
    finally:
        ens.close()
