"""Sums read back through pinned memory by the last workgroup to finish: one
workgroup and many, repeated, from several threads at once."""

import ctypes
import threading

import numpy as np
import pytest

import ember_amd as em
from ember_amd import capi, loss
from ember_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1, 255, 256, 257, 1000, 65536, 262143, 262145, 1 << 20, 5000003])
def test_sum_of_every_workgroup_count(size):
    x = np.random.default_rng(size).standard_normal(size, dtype=np.float32)
    t = Tensor(x)
    first = em.sum(t)
    # Doubles throughout and one rounding to fp32.
    exact = x.astype(np.float64).sum()
    assert first == pytest.approx(exact, rel=2.0 ** -23, abs=1e-9 * size)
    for _ in range(20):
        assert em.sum(t) == first


def test_threads_get_their_own_sums():
    rng = np.random.default_rng(0)
    xs = [Tensor(rng.standard_normal(n, dtype=np.float32)) for n in (3, 70000, 300000, 1500000)]
    logits = [Tensor(rng.standard_normal((n, 50), dtype=np.float32)) for n in (2, 700, 20000)]
    ts = [Tensor(np.full(x.shape, 0.02, np.float32)) for x in logits]
    want = [em.sum(x) for x in xs] + [loss.CrossEntropyLoss()(x, t) for x, t in zip(logits, ts)]
    bad = []

    def work():
        for _ in range(50):
            got = [em.sum(x) for x in xs] + [loss.CrossEntropyLoss()(x, t) for x, t in zip(logits, ts)]
            if got != want:
                bad.append(got)

    threads = [threading.Thread(target=work) for _ in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, (bad[0], want)


@pytest.mark.parametrize("which", ["mse_loss", "cross_entropy_loss"])
def test_tensors_are_whole_when_the_call_returns(which):
    """The gradient is read at once on a stream that the null stream does not
    order, as the call is documented to synchronise."""
    rows, classes = 4096, 1024
    L, rng = capi.lib(), np.random.default_rng(0)
    x, t = (rng.random((rows, classes), dtype=np.float32) for _ in range(2))
    e = np.exp(x.astype(np.float64))
    want = 2 * (x - t) if which == "mse_loss" else e / e.sum(-1, keepdims=True) - t
    dx, dt, zero = (capi.DeviceArray.from_numpy(a) for a in (x, t, np.zeros_like(x)))
    p, grad, copy = (capi.DeviceArray(x.shape) for _ in range(3))
    args = (rows * classes, ctypes.c_float(2.0)) if which == "mse_loss" else (rows, classes, 1.0)
    ptrs = [ctypes.c_void_p(a.ptr) for a in ((dx, dt, grad) if which == "mse_loss" else (dx, dt, p, grad))]
    side, total, to_device = ctypes.c_void_p(), ctypes.c_float(), 3  # hipMemcpyDeviceToDevice
    n, cp = ctypes.c_size_t(grad.nbytes), lambda a: ctypes.c_void_p(a.ptr)  # noqa: E731
    assert L.hipStreamCreateWithFlags(ctypes.byref(side), 1) == 0  # hipStreamNonBlocking
    for _ in range(20):
        assert L.hipMemcpy(cp(grad), cp(zero), n, to_device) == 0
        assert L.hipDeviceSynchronize() == 0
        capi.check(getattr(L, which)(*ptrs, *args, ctypes.byref(total)), which)
        assert L.hipMemcpyAsync(cp(copy), cp(grad), n, to_device, side) == 0
        assert L.hipStreamSynchronize(side) == 0
        # A few fp32 roundings of values up to 2, and expf's.
        np.testing.assert_allclose(copy.numpy(), want, rtol=0, atol=1e-6)
    assert L.hipStreamDestroy(side) == 0
