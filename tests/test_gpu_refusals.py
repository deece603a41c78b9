"""Calls that fail leave the handle, and the thread, as their callers may rely on: later calls work."""
import ctypes

import numpy as np
import pytest

from poe2d_amd import _abi
from poe2d_amd.mlp import DeviceArray, Network
from poe2d_amd.solver import ReceiverSpec, Solver, SourceSpec

from .helpers import small_problem

pytestmark = pytest.mark.gpu

TOO_LARGE = (1 << 33, 1 << 10)  # 32 TB of floats


def shot(nt=9):
    rec = ReceiverSpec(ix=np.arange(20, 100, 7), iz=np.full(12, 50))
    src = SourceSpec(kind=_abi.SRC_PRESSURE_DGAUSS, ix=60, iz=60, amp=1e6)
    return small_problem(src=src, rec=rec, nt=nt)


def refused(f):
    with pytest.raises(_abi.Poe2dError) as e:
        f()
    assert e.value.status == _abi.POE2D_E_NOMEM


def test_a_refused_allocation_is_not_reported_by_the_next_call():
    with Solver(shot()) as s, Network([4, 64, 64], max_batch=32) as net:
        x = np.ones((3, 4), np.float32)
        y = net.predict(x)[0]
        for call in (s.reset, lambda: s.run(3), lambda: net.predict(x), lambda: Network([4, 8], max_batch=32).close()):
            refused(lambda: DeviceArray(TOO_LARGE))
            call()
        refused(lambda: Network([1 << 20, 1 << 26], max_batch=32))
        assert np.array_equal(net.predict(x)[0], y)
        s.run(1)
        assert s.step_count() == 4


def test_receivers_whose_traces_do_not_fit_leave_the_handle_without_receivers():
    prob = shot()
    with Solver(prob) as s:
        s.run()
        ref = s.seismograms()
        # 25 TB of traces, at more positions than the handle had
        far = ReceiverSpec(ix=np.tile(np.arange(100), 10), iz=np.repeat(np.arange(10), 100), nsamp=2 ** 31 - 1)
        refused(lambda: s.set_receivers(far))
        s.reset()
        s.run(5)
        assert s.step_count() == 5 and np.isfinite(s.snapshot("vx")).all()
        s.reset()
        s.set_receivers(prob.receivers)
        s.run()
        assert np.array_equal(s.seismograms(), ref)


def test_a_copy_that_the_runtime_refuses_is_not_reported_by_the_next_call():
    with Solver(shot()) as s, Network([4, 64, 64], max_batch=32) as net:
        x = np.ones((3, 4), np.float32)
        y = net.predict(x)[0]
        short = DeviceArray((10, 4096))
        host = np.zeros((100, 4096), np.float32)
        for call in (s.reset, lambda: s.run(3), lambda: net.predict(x)):
            assert s._lib.poe2d_copy(ctypes.c_void_p(short.ptr), ctypes.c_void_p(host.ctypes.data),
                                     ctypes.c_size_t(host.nbytes)) == _abi.POE2D_E_HIP
            call()
        assert np.array_equal(net.predict(x)[0], y)


@pytest.mark.parametrize("held", [10, 70])
def test_a_prediction_into_device_memory_that_is_too_short_is_refused(held):
    """Batches of 64 rows: the first, or the second, does not fit."""
    rows = 100
    rng = np.random.default_rng(5)
    with Network([8, 64, 4096], members=2, max_batch=64) as net:
        x = rng.standard_normal((rows, 8)).astype(np.float32)
        ref, spread = net.predict(x)
        short, whole = DeviceArray((held, 4096)), DeviceArray((rows, 4096))
        fp = _abi.c_float_p
        args = net._h, rows, x.ctypes.data_as(fp)
        assert net._lib.poe2d_mlp_predict(*args, ctypes.cast(ctypes.c_void_p(short.ptr), fp), None) == _abi.POE2D_E_HIP
        got, s = net.predict(x, out=whole)
        assert np.array_equal(got.to_host(), ref) and np.array_equal(s, spread)
