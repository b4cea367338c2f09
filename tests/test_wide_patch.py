"""A patch whose rows are too long for 32-bit offsets in the stage tiles (2^32
bytes over 22 rows: 24.4 million cells), which takes the 64-bit form of the
stage: a uniform state with structure at both ends gives at each end, bit for
bit, what a patch of 400 columns gives (32-bit offsets), with the same dt, and
nothing moves in between.  The state is 25 GB on the host, twice while it is
uploaded, and 73 GB on the device."""
import ctypes
import os

import numpy as np
import pytest

from sac_amd import problems

pytestmark = pytest.mark.gpu

NY, STEPS, M = 6, 2, 96  # M: columns compared at each end


def _state(g0):
    w = np.zeros((13, NY + 4, g0))
    w[0], w[4] = 1.0, 1.5
    rng = np.random.default_rng(3)
    w[:8, :, 2:42] += 0.05 * rng.standard_normal((8, NY + 4, 40))
    w[:8, :, g0 - 42:g0 - 2] += 0.05 * rng.standard_normal((8, NY + 4, 40))
    return w


def _run(nx):
    from sac_amd import batch
    L = batch._lib()
    w = _state(nx + 4)
    dx = np.full(nx + NY + 8, 0.01)
    n = np.array([nx, NY], dtype=np.int32)
    eq = np.array([5.0 / 3.0, 0, 0, 0, 0, 1.0])
    h = ctypes.c_void_p()
    batch._check(L.sac_batch_init_nd(2, 1, batch._ip(n), 13, batch._dp(w), batch._dp(dx),
                                     batch._dp(eq), 6, problems.NU, 0.3, 1e9, 1000,
                                     ctypes.byref(h)))
    try:
        done = ctypes.c_longlong()
        batch._check(L.sac_batch_run(h, -1, STEPS, ctypes.byref(done)))
        batch._check(L.sac_batch_download(h, batch._dp(w)))
        t = np.zeros(1)
        batch._check(L.sac_batch_status(h, batch._dp(t), None, None))
    finally:
        L.sac_batch_free(h)
    return w, t[0]


def test_rows_beyond_32_bit_offsets():
    nx = 24_500_000
    assert (nx + 4) * 8 * 22 >= 2 ** 32
    if os.sysconf("SC_AVPHYS_PAGES") * os.sysconf("SC_PAGE_SIZE") < 100 << 30:
        pytest.skip("needs 100 GB of host memory")
    small, ts = _run(400)
    wide, tw = _run(nx)
    assert tw == ts > 0.0
    np.testing.assert_array_equal(wide[:, :, :M], small[:, :, :M])
    np.testing.assert_array_equal(wide[:, :, -M:], small[:, :, -M:])
    assert np.abs(small - _state(404)).max() > 1e-2
    mid = wide[:8, 2:-2, M:-M:9973]
    np.testing.assert_array_equal(mid, np.broadcast_to(mid[:, :1, :1], mid.shape))
