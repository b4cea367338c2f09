"""Transfers, saves and allocations on a stand-in for the HIP runtime
(hip_host.c): what the library does when an allocation or a launch fails, and
what it leaves behind.  No GPU."""
import pytest

from tests import hip_host


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hip_host.build(tmp_path_factory.mktemp("hip_host"))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_save_keeps_its_background(stub, precision):
    """save_end gives the state at save_begin, the background too, whatever
    was uploaded or filled in between."""
    hip_host.run(stub, f"""
        p = state_problem((31, 27, 35))
        dev = device.Device(p, precision={precision!r})
        want = p.w.copy()
        if {precision!r} == "mixed":
            want[:8] = want[:8].astype(np.float32)
        dev.upload(p.w)
        dev.save_begin()
        dev.upload(-p.w)
        np.testing.assert_array_equal(dev.save_end(), want)
        dev.upload(p.w)
        dev.save_begin()
        dev.getboundary()
        np.testing.assert_array_equal(dev.save_end(), want)
        # a later save has the background of its own time
        dev.upload(-p.w)
        dev.save_begin()
        np.testing.assert_array_equal(dev.save_end(), -want)
    """)
