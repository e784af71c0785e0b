"""The one-pass cross-entropy (cross_entropy_loss) at the edges of its row
forms, against float64, and what it does with infinities next to the composed
operators."""

import ctypes as C

import numpy as np
import pytest

from ember_amd import capi, loss
from ember_amd.capi import DeviceArray
from ember_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


def _case(rows, classes, seed):
    rng = np.random.default_rng(seed)
    x = 3 * rng.standard_normal((rows, classes), dtype=np.float32)
    t = rng.random((rows, classes), dtype=np.float32)
    return x, t / t.sum(-1, keepdims=True)


def _ref(x, t, n):
    s = x.astype(np.float64) - x.max(-1, keepdims=True)
    lp = s - np.log(np.exp(s).sum(-1, keepdims=True))
    return (t * lp).sum(), np.exp(lp), (np.exp(lp) - t) / n


def _check(value, probs, grad, x, t, n):
    # p: expf, logf and two fp32 roundings of a log-probability of up to ~25
    # (2^-20 absolute), so 4e-6 relative; the gradient's (p - t) adds 2^-24 of
    # the larger of the two.
    rv, rp, rg = _ref(x, t, n)
    assert value == pytest.approx(rv, rel=2e-6)
    np.testing.assert_allclose(probs, rp, rtol=4e-6, atol=1e-30)
    np.testing.assert_allclose(grad * n, rg * n, rtol=4e-6, atol=4e-6 * max(rp.max(), t.max()))


@pytest.mark.parametrize("rows,classes", [
    (1, 1), (5, 2), (33, 10), (16, 16), (17, 17), (9, 32), (5, 33), (7, 64), (6, 65), (5, 127), (5, 129), (4, 256),
    (4, 260), (3, 255), (3, 512), (3, 516), (3, 513), (8300, 24), (33000, 12), (9, 1000), (9, 1001), (5, 1024),
    (5, 1028), (4, 1025), (4, 2048), (4, 2052), (3, 4096), (3, 4095), (3, 4100), (2, 10001), (2100, 1030),
])
def test_sizes(rows, classes):
    x, t = _case(rows, classes, rows + classes)
    ce = loss.CrossEntropyLoss()
    value = ce(Tensor(x), Tensor(t))
    _check(-value * rows, ce.probs.to_np(), ce.backward().to_np(), x, t, rows)


@pytest.mark.parametrize("classes", [64, 1000, 1024, 2048])
@pytest.mark.parametrize("which", range(4))
def test_pointers_off_16_bytes(classes, which):
    """One of the four arrays 4 bytes off: scalar loads."""
    rows = 5
    x, t = _case(rows, classes, classes)
    L = capi.lib()
    off = [4 * (which == i) for i in range(4)]
    bufs = [DeviceArray((rows * classes + 1,)) for _ in range(2)]
    total = C.c_float()
    ins = []
    for o, v in zip(off, (x, t)):
        full = np.zeros(rows * classes + 1, np.float32)
        full[o // 4:o // 4 + rows * classes] = v.ravel()
        ins.append(DeviceArray.from_numpy(full))
    ptrs = [b.ptr + o for b, o in zip(ins + bufs, off)]
    capi.check(L.cross_entropy_loss(*ptrs, rows, classes, float(rows), C.byref(total)), "cross_entropy_loss")
    probs, grad = (b.numpy()[o // 4:o // 4 + rows * classes].reshape(rows, classes) for b, o in zip(bufs, off[2:]))
    _check(total.value, probs, grad, x, t, rows)


@pytest.mark.parametrize("classes", [10, 100, 1000, 5000])
def test_infinities_as_the_composed_operators(classes):
    """-inf logits (probability 0, and 0 * -inf in the sum), +inf, NaN and
    the lowest number: the same values as the composition, which a broadcast
    target of the same content takes."""
    x, t = _case(6, classes, 3)
    x[0, 1] = -np.inf
    x[1, 2] = np.inf
    x[2, 3] = np.nan
    x[3, 4] = np.finfo(np.float32).min
    x[4] = -np.inf
    t[:] = t[0]
    fused, composed = loss.CrossEntropyLoss(), loss.CrossEntropyLoss()
    a = fused(Tensor(x), Tensor(t))
    b = composed(Tensor(x), Tensor(t[:1]))
    assert fused.grad is not None and composed.grad is None
    assert np.isnan(a) == np.isnan(b) and np.isnan(a)
    for got, want in ((fused.probs, composed.probs), (fused.backward(), composed.backward())):
        np.testing.assert_allclose(got.to_np(), want.to_np(), rtol=4e-6, atol=1e-7)


def test_refuses_what_it_cannot_take():
    L = capi.lib()
    total = C.c_float()
    for rows in (-1, 2):
        with pytest.raises(Exception):
            capi.check(L.cross_entropy_loss(None, None, None, None, rows, 4, 1.0, C.byref(total)), "cross_entropy_loss")
    assert L.cross_entropy_loss(None, None, None, None, 0, 4, 1.0, C.byref(total)) == 0


def test_most_rows():
    """2^31 - 1 rows of one class: the row indexes ahead of the last pass 2^31."""
    rows, part = 2 ** 31 - 1, 1 << 20
    L = capi.lib()
    x, t, probs, grad = (DeviceArray((rows,)) for _ in range(4))
    for a in (x, t, probs, grad):
        L.hipMemset(C.c_void_p(a.ptr), 0, C.c_size_t(a.nbytes))
    total = C.c_float(1)
    capi.check(L.cross_entropy_loss(x.ptr, t.ptr, probs.ptr, grad.ptr, rows, 1, 2.0, C.byref(total)),
               "cross_entropy_loss")
    assert total.value == 0
    for a, want in ((probs, 1), (grad, 0.5)):
        for first in (0, rows // 2, rows - part):
            got = np.empty(part, np.float32)
            L.copy_from_device(got.ctypes.data, a.ptr + 4 * first, got.nbytes)
            assert (got == want).all()


@pytest.mark.parametrize("cls", [loss.CrossEntropyLoss, loss.MSELoss])
def test_each_backward_gives_a_gradient_of_its_own(cls):
    """What a caller does to the tensor it got, in place or through its
    buffer, does not reach the next call's."""
    x, t = _case(7, 50, 11)
    fn = cls()
    fn(Tensor(x), Tensor(t))
    first = fn.backward()
    want = first.to_np()
    first *= 3.0
    second = fn.backward()
    np.testing.assert_array_equal(second.to_np(), want)
    L = capi.lib()
    assert L.hipMemset(C.c_void_p(second._core.data_ptr), 0, C.c_size_t(4 * x.size)) == 0
    assert not second.to_np().any()
    np.testing.assert_array_equal(fn.backward().to_np(), want)


@pytest.mark.parametrize("n", [1e-40, 1e-38, -2.0, 0.25, 3e38, 0.0, np.inf, np.nan])
def test_any_divisor(n):
    """The C entry's n: (probs - target) / n as fp32 divides, also where 1 / n
    is denormal or infinite."""
    rows, classes = 9, 100
    x, t = _case(rows, classes, 12)
    t[:] = 0
    t[:, 3] = 1
    L, total = capi.lib(), C.c_float()
    dx, dt = DeviceArray.from_numpy(x), DeviceArray.from_numpy(t)
    p, g = DeviceArray(x.shape), DeviceArray(x.shape)
    capi.check(L.cross_entropy_loss(dx.ptr, dt.ptr, p.ptr, g.ptr, rows, classes, n, C.byref(total)), "cross_entropy_loss")
    with np.errstate(all="ignore"):
        want = (p.numpy() - t) / np.float32(n)
    # Equal but for the sign of a zero.
    np.testing.assert_array_equal(g.numpy() + np.float32(0), want + np.float32(0))
    assert total.value == pytest.approx(_ref(x, t, 1)[0], rel=2e-6)
