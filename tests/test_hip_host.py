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


@pytest.mark.parametrize("n", [(70, 61, 64), (300001,)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("where", [1, 2])
def test_copy_reports_a_failed_launch(stub, n, precision, where):
    """A copy kernel that cannot be launched fails the call, whichever thread
    launched it (a state of several chunks)."""
    hip_host.run(stub, f"""
        p = state_problem({n!r})
        dev = device.Device(p, precision={precision!r})
        dev.upload(p.w)
        assert knob("threads").value > 0  # chunks went over other threads
        knob("fail_launch").value = {where}
        for call in (lambda: dev.upload(p.w), dev.download,
                     lambda: dev.upload_slot(1, p.w), lambda: dev.download_slot(1)):
            try:
                call()
            except device.SacError as e:
                assert "failed" in str(e), e
            else:
                raise AssertionError("reported as done")
        knob("fail_launch").value = 0
        dev.upload(p.w)
        np.testing.assert_array_equal(dev.download()[8:], p.w[8:])
    """)


@pytest.mark.parametrize("n", [(800,), (300001,)])
def test_copy_is_not_failed_by_an_earlier_error(stub, n):
    """An error that some other call of the program left behind is not a
    copy's, and the copy leaves it where it is."""
    hip_host.run(stub, f"""
        p = state_problem({n!r})
        dev = device.Device(p)
        for call in (lambda: dev.upload(p.w), dev.download, lambda: dev.upload_slot(1, p.w)):
            assert hip.hipMemcpy(None, None, 0, 0) == 1
            call()
            assert hip.hipGetLastError() == 1
    """)


@pytest.mark.parametrize("where", [1, 2])
def test_ensemble_download_reports_a_failed_launch(stub, where):
    hip_host.run(stub, f"""
        ens = batch.Ensemble([state_problem((n,)) for n in (20000, 30000, 40000, 50000, 9000)] * 3)
        ens.download()
        assert knob("threads").value > 0
        knob("fail_launch").value = {where}
        try:
            ens.download()
        except device.SacError as e:
            assert "failed" in str(e), e
        else:
            raise AssertionError("reported as done")
    """)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("what,n", [("fail_malloc", 1), ("fail_event", 1), ("fail_event", 2),
                                    ("fail_pinned", 1)])
def test_save_after_a_failed_allocation(stub, precision, what, n):
    """A save that cannot get its buffers returns an error; one that can,
    later, is a save like any other."""
    hip_host.run(stub, f"""
        p = state_problem((16, 9, 8))
        want = p.w.copy()
        if {precision!r} == "mixed":
            want[:8] = want[:8].astype(np.float32)
        dev = device.Device(p, precision={precision!r})
        dev.upload(p.w)
        dev.download()
        before = dev.memory()
        knob({what!r}).value = {n}
        for _ in range({3 if what == "fail_pinned" else 1}):
            try:
                dev.save_begin()
            except device.SacError:
                pass
            else:
                raise AssertionError("no error")
        knob({what!r}).value = 0
        dev.save_begin()
        assert dev.save_ready()
        np.testing.assert_array_equal(dev.save_end(), want)
        assert knob("null_stores").value == 0
        dev.save_begin()
        np.testing.assert_array_equal(dev.save_end(), want)
        assert dev.memory() == before + 20 * 13 * 12 * 8 * {4 if precision == "mixed" else 8}
        dev.close()
        assert knob("pinned_now", ctypes.c_size_t).value == 0
    """)


def test_reported_errors_are_not_reported_again(stub):
    """An allocation that failed is an error of the call that made it, not of
    the next call of this library or of the program."""
    hip_host.run(stub, """
        p = state_problem((16, 9, 8))
        knob("fail_malloc").value = 3
        try:
            device.Device(p)
        except device.SacError as e:
            assert "hipMalloc" in str(e)
        else:
            raise AssertionError("no error")
        assert hip.hipGetLastError() == 0
        dev = device.Device(p)
        dev.upload(p.w)
        for what in ("fail_malloc", "fail_event", "fail_pinned"):
            knob(what).value = 1
            try:
                dev.save_begin()
            except device.SacError:
                pass
            else:
                raise AssertionError("no error")
            knob(what).value = 0
            dev.getboundary()
            dev.synchronize()
            dev.save_begin()
            dev.save_end()
            dev.close()
            dev = device.Device(p)
            dev.upload(p.w)
        # a small copy without pinned memory
        t = state_problem((50,))
        small = device.Device(t)
        knob("fail_pinned").value = 1
        try:
            small.upload(t.w)
        except device.SacError:
            pass
        assert hip.hipGetLastError() == 0
        knob("fail_pinned").value = 0
        tubes = [state_problem((n,)) for n in (20, 30)]
        knob("fail_malloc").value = 2
        try:
            batch.Ensemble(tubes)
        except device.SacError:
            pass
        assert hip.hipGetLastError() == 0
    """)


def test_copies_leave_the_current_device(stub):
    """A thread whose current device is not the handle's keeps it through the
    copies, as through those of one buffer."""
    hip_host.run(stub, """
        cur = ctypes.c_int()
        p = state_problem((70, 61, 64))
        dev = device.Device(p)
        ens = batch.Ensemble([state_problem((n,)) for n in (20000, 30000, 40000, 50000)])
        assert hip.hipSetDevice(1) == 0
        for call in (lambda: dev.upload(p.w), dev.download, lambda: dev.upload_slot(1, p.w),
                     lambda: dev.download_slot(1), ens.download):
            call()
            hip.hipGetDevice(ctypes.byref(cur))
            assert cur.value == 1, cur.value
        np.testing.assert_array_equal(dev.download(), p.w)
    """)


@pytest.mark.parametrize("n", [(800,), (300001,), (61, 47), (70, 61, 64)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("where", [1, 2])
def test_copies_without_pinned_memory(stub, n, precision, where):
    """Pinned memory makes copies fast and is no condition for them: with none
    at all (1), or none for the worker threads (2), states go up and down."""
    hip_host.run(stub, f"""
        knob("fail_pinned").value = {where}
        p = state_problem({n!r})
        want = p.w.copy()
        if {precision!r} == "mixed":
            want[:8] = want[:8].astype(np.float32)
        dev = device.Device(p, precision={precision!r})
        dev.upload(p.w)
        np.testing.assert_array_equal(dev.download(), want)
        other = state_problem({n!r}, seed=6).w
        dev.upload_slot(1, other)
        want[:8] = other[:8].astype(np.float32) if {precision!r} == "mixed" else other[:8]
        np.testing.assert_array_equal(dev.download_slot(1), want)
        dev.getboundary()
        dev.getdt_special(1.0)
        assert dev.maxviscoef == 0.0
        assert hip.hipGetLastError() == 0
    """)


@pytest.mark.parametrize("ndim", [1, 2])
def test_ensemble_download_without_pinned_memory(stub, ndim):
    hip_host.run(stub, f"""
        knob("fail_pinned").value = 1
        probs = [state_problem((n,) if {ndim} == 1 else (n, 60 - n // 2)) for n in (6, 33, 90)]
        ens = batch.Ensemble(probs)
        for got, p in zip(ens.download(), probs):
            np.testing.assert_array_equal(got, p.w)
        assert hip.hipGetLastError() == 0
    """)


def test_ensemble_download_pins_no_more_than_its_buffers(stub):
    """However large the members are: eight buffers of 4 MB."""
    hip_host.run(stub, """
        ens = batch.Ensemble([state_problem((n,)) for n in (200000, 300, 150000, 90000)])
        knob("pinned_peak", ctypes.c_size_t).value = 0
        knob("pinned_most", ctypes.c_size_t).value = 0
        ens.download()
        assert 0 < knob("pinned_most", ctypes.c_size_t).value <= 4 << 20
        assert knob("pinned_peak", ctypes.c_size_t).value <= 8 * (4 << 20)
        assert knob("pinned_now", ctypes.c_size_t).value == 0
    """)


def test_ensemble_download_allocates_nothing_on_the_device(stub):
    hip_host.run(stub, """
        probs = [state_problem((n,)) for n in (20000, 300)]
        ens = batch.Ensemble(probs)
        before = ens.memory()
        knob("fail_malloc").value = 1
        ens.download()
        assert ens.memory() == before and knob("fail_malloc").value == 1
    """)


@pytest.mark.parametrize("ndim,n", [(1, 1), (2, 1), (2, 2)])
def test_shape_whose_tables_cannot_be_allocated(stub, ndim, n):
    """The ensemble goes on with the tables it has."""
    hip_host.run(stub, f"""
        probs = [state_problem((n,) if {ndim} == 1 else (n, 60 - n // 2)) for n in (6, 33, 90)]
        ens = batch.Ensemble(probs)
        ens.run(steps_per_graph=-1, max_steps=1)
        assert knob("freed_used").value == 0
        was = ens.shape()
        knob("fail_malloc").value = {n}
        try:
            ens.set_shape(0)
        except device.SacError:
            assert ens.shape() == was
        else:
            assert knob("fail_malloc").value > 0  # it takes fewer allocations
        knob("fail_malloc").value = 0
        ens.run(steps_per_graph=-1, max_steps=1)
        assert knob("freed_used").value == 0
        ens.set_shape(0)
        ens.run(steps_per_graph=-1, max_steps=1)
        assert knob("freed_used").value == 0
    """)


@pytest.mark.parametrize("n", [1, 3, 7, 9])
def test_closure_that_cannot_be_allocated(stub, n):
    """It is not there, its memory is given back, and it can be asked for
    again."""
    hip_host.run(stub, f"""
        from sac_amd import closure
        p = state_problem((16, 9, 8))
        dev = device.Device(p)
        before = dev.memory()
        knob("fail_malloc").value = {n}
        try:
            closure.Closure(dev, capacity=1000)
        except device.SacError as e:
            assert "hipMalloc" in str(e), e
        else:
            raise AssertionError("no error")
        assert dev.memory() == before
        L = closure._lib()
        assert L.sac_closure_enable(dev.handle, 1, 0.1) == 1  # not initialised
        closure.Closure(dev, capacity=1000)
        assert dev.memory() > before
        assert L.sac_closure_enable(dev.handle, 1, 0.1) == 0
    """)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_copies_without_host_memory(stub, precision):
    """Where the host has no memory left for a thread or a list, a copy is
    slower or an error, never an exception out of a C entry point."""
    hip_host.run(stub, f"""
        p = state_problem((70, 61, 64))
        dev = device.Device(p, precision={precision!r})
        dev.upload(p.w)
        want = dev.download()
        dev.save_begin()
        dev.save_end()
        ens = batch.Ensemble([state_problem((n,)) for n in (20000, 30000, 40000, 50000)])
        ens.download()

        def save():
            dev.save_begin()
            return dev.save_end()

        def first_save():  # copies the background too
            dev.upload(want)
            knob("fail_new").value = n
            return save()

        lost = done = 0
        for call in (lambda: dev.upload(p.w), dev.download, ens.download, save, first_save):
            for n in range(1, 20):
                knob("fail_new").value = n
                try:
                    got = call()
                    if knob("fail_new").value == 0:
                        done += 1
                    if call not in (ens.download,) and got is not None:
                        np.testing.assert_array_equal(got, want)
                except device.SacError as e:
                    assert "host memory" in str(e), e
                    lost += 1
                knob("fail_new").value = 0
        assert lost > 0 and done > 0
        dev.upload(p.w)
        np.testing.assert_array_equal(dev.download(), want)
    """)
