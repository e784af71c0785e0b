"""The split-bf16 GEMM where it can go wrong: tile edges and short last k-slabs
of each tile shape and orientation, operands that do not start on 16 bytes,
values the split cannot carry (infinities, NaN, magnitudes next to the largest
float), elements of every magnitude beside larger ones, extents up to 2^31 - 1,
and its error against float64 next to the fp32 chain's."""

import ctypes as C

import numpy as np
import pytest

import gpu_helpers as G
from ember_amd import capi

pytestmark = pytest.mark.gpu


def _u(shape, seed):
    return np.random.default_rng(seed).uniform(-1, 1, shape).astype(np.float32)


def _stored(x, trans):
    return np.ascontiguousarray(x.T) if trans else x


def _bound(a, b):
    """6 roundings per 16 products of partial sums of at most |a||b|, and the
    part products left out: mid up to 2^-8 and lo up to 2^-17 of an element,
    so 2 * 2^-25 + 2^-34 of |a||b|, rounded up."""
    k = a.shape[1]
    mag = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    return (0.375 * k + 8) * 2.0 ** -24 * mag + 2.0 ** -23 * mag


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("n,k,m", [
    (1, 1, 1), (64, 32, 64), (65, 33, 63), (63, 31, 65), (3, 64, 200),     # 64 x 64 tiles, one to two slabs
    (129, 1030, 127), (640, 97, 1537),                                     # splits; ragged in all three
    (2500, 130, 1900), (4096, 15, 4097), (4097, 47, 4095),                 # 128 and 256 tiles with remainders
])
def test_shapes_and_orientations(n, k, m, ta, tb):
    a, b = _u((n, k), n + k), _u((k, m), m)
    got = G.gemm_ex(_stored(a, ta), _stored(b, tb), ta, tb)
    rows = np.unique(np.r_[0, n - 1, np.random.default_rng(0).integers(0, n, 40)])
    ref = a[rows].astype(np.float64) @ b.astype(np.float64)
    assert (np.abs(got[rows] - ref) <= _bound(a[rows], b)).all()


@pytest.mark.parametrize("offset", [1, 2, 3])
def test_operands_off_16_bytes(offset):
    n, k, m = 70, 100, 130
    a, b = _u((n, k), 1), _u((k, m), 2)
    bufs = [capi.DeviceArray((x.size + 4,), np.r_[np.zeros(offset, np.float32), x.ravel(),
                                                  np.zeros(4 - offset, np.float32)]) for x in (a, b)]
    out = capi.DeviceArray((n * m + 4,))
    L = capi.lib()
    L.matmul(bufs[0].ptr + 4 * offset, bufs[1].ptr + 4 * offset, out.ptr + 4 * offset, n, m, k)
    capi.check(what="matmul")
    got = out.numpy()[offset:offset + n * m].reshape(n, m)
    assert (np.abs(got - a.astype(np.float64) @ b) <= _bound(a, b)).all()


@pytest.mark.parametrize("n,k,m", [(100, 70, 90), (600, 500, 700), (4096, 40, 4096)])
def test_infinities_and_nan_follow_ieee(n, k, m):
    """An infinite element gives +-inf or NaN exactly where fp32 products and
    sums do, and leaves every other element as it is."""
    a, b = _u((n, k), 3), _u((k, m), 4)
    a[n // 2, 3], a[n - 1, k - 1], b[5, m // 3] = np.inf, -np.inf, -np.inf
    b[3, 7] = 0.0          # inf * 0
    a[1, 2] = np.nan
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    got = G.gemm_ex(a, b)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)].astype(np.float32))
    ok = np.isfinite(ref)
    fa, fb = np.where(np.isfinite(a), a, 0), np.where(np.isfinite(b), b, 0)
    assert (np.abs(got - ref)[ok] <= _bound(fa, fb)[ok]).all()


def test_magnitudes_next_to_the_largest_float():
    """The largest finite floats round up to infinity in bf16; their products
    with small factors are finite."""
    n, k, m = 80, 48, 70
    a, b = _u((n, k), 5), _u((k, m), 6) * np.float32(2.0 ** -20)
    a[4] = np.finfo(np.float32).max
    a[9, :] = np.finfo(np.float32).min
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert (np.abs(G.gemm_ex(a, b) - ref) <= _bound(a, b)).all()


@pytest.mark.parametrize("exponent", [-99, -101, -110, -125])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_tiny_rows_keep_their_precision(exponent, ta, tb):
    """Rows of a and columns of b below what three bf16 parts can hold without
    a scale; the other operand brings the results back into range."""
    n, k, m = 90, 200, 75
    a, b = _u((n, k), 7), _u((k, m), 8) * np.float32(2.0 ** 60)
    a[10:20] *= np.float32(2.0 ** exponent)
    b[:, 30] *= np.float32(2.0 ** (exponent - 60))
    ref = a.astype(np.float64) @ b.astype(np.float64)
    got = G.gemm_ex(_stored(a, ta), _stored(b, tb), ta, tb)
    err, bound = np.abs(got - ref), _bound(a, b) + 2.0 ** -149 * k
    assert (err <= bound).all()


@pytest.mark.parametrize("n,k,m,fp32_chain", [(4096, 1024, 4096, 5.7e-7), (1024, 8192, 1024, 4.1e-7),
                                               (8192, 1024, 1024, 4.0e-7), (197, 333, 250, 3.2e-7)])
def test_error_no_larger_than_the_fp32_instructions(n, k, m, fp32_chain):
    """Relative 2-norm error against float64, U(-1, 1) operands: below what
    the kernels on the fp32 matrix instruction measured at these shapes."""
    a, b = _u((n, k), 9), _u((k, m), 10)
    got = G.gemm_ex(a, b)
    rows = np.arange(0, n, max(1, n // 64))
    ref = a[rows].astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(got[rows] - ref) / np.linalg.norm(ref) <= fp32_chain


@pytest.mark.parametrize("n,k,m,fp32_chain", [(4096, 1024, 1024, 5.5e-7), (4096, 4096, 4096, 1.12e-6), (1024, 8192, 512, 4.5e-7)])
def test_sums_over_rows_and_columns_are_unbiased(n, k, m, fp32_chain):
    """A rounding of one direction in the matrix core would add up over the
    rows of a column (a bias gradient): held to what the fp32 instruction's
    sums measured (1.3e-5 without the row and column signs at 4096^3)."""
    a, b = _u((n, k), 11), _u((k, m), 12)
    got = G.gemm_ex(a, b).astype(np.float64)
    for axis, ref in ((0, a.sum(0, dtype=np.float64) @ b), (1, a.astype(np.float64) @ b.sum(1, dtype=np.float64))):
        assert np.linalg.norm(got.sum(axis) - ref) / np.linalg.norm(ref) <= 1.2 * fp32_chain


def test_zero_products_give_positive_zero():
    a, b = _u((70, 40), 13), np.zeros((40, 90), np.float32)
    assert not np.signbit(G.gemm_ex(a, b)).any()


@pytest.mark.parametrize("k", [1431655765, 1500000001, 2 ** 31 - 1])
def test_longest_sums(k):
    """A dot product whose k, in chunks and slabs, passes 2^31: zeros but for
    whole numbers at the ends, about every split's likely ends and 2^30."""
    at = np.unique(np.clip(np.r_[0:40, k - 40:k, 2 ** 30 - 20:2 ** 30 + 20,
                                 np.concatenate([np.arange(-2, 34) + k * z // 64 for z in range(64)])], 0, k - 1))
    a = capi.DeviceArray((k,))
    one, out = np.ones(1, np.float32), capi.DeviceArray((1,))
    L = capi.lib()
    assert L.hipMemset(C.c_void_p(a.ptr), 0, C.c_size_t(a.nbytes)) == 0
    for i in at:
        L.copy_to_device(a.ptr + 4 * int(i), one.ctypes.data, 4)
    for ta, tb in ((0, 0), (1, 1)):
        capi.check(L.gemm_ex(a.ptr, a.ptr, out.ptr, 1, 1, 1, k, ta, tb, None, None, None, 0), "gemm_ex")
        assert out.numpy()[0] == len(at)


@pytest.mark.parametrize("size", [2 ** 30 + 1, 1100000000, 2 ** 31 - 200, 2 ** 31 - 1])
@pytest.mark.parametrize("rows", [True, False])
def test_longest_outputs(size, rows):
    """One column or row of more tiles than one grid holds threads for."""
    L = capi.lib()
    a, b, out = capi.DeviceArray((size,)), capi.DeviceArray((1,), np.full(1, 3, np.float32)), capi.DeviceArray((size,))
    n, m = (size, 1) if rows else (1, size)
    assert L.hipMemset(C.c_void_p(a.ptr), 0x40, C.c_size_t(a.nbytes)) == 0
    assert L.hipMemset(C.c_void_p(out.ptr), 0, C.c_size_t(out.nbytes)) == 0
    x, y = (a, b) if rows else (b, a)
    for k, want in ((1, 3 * np.full(1, 0x40404040, np.uint32).view(np.float32)[0]), (0, 0)):
        capi.check(L.gemm_ex(x.ptr, y.ptr, out.ptr, 1, n, m, k, 0, 0, None, None, None, 0), "gemm_ex")
        part = np.empty(min(size, 1 << 22), np.float32)
        for first in (0, size // 2, 2 ** 30 - len(part), size - len(part)):
            L.copy_from_device(part.ctypes.data, out.ptr + 4 * first, part.nbytes)
            assert (part == want).all()


@pytest.mark.parametrize("small,large", [(-95, 60), (-112, 90), (-120, 100), (-126, 100), (-135, 110), (-145, 100)])
@pytest.mark.parametrize("n,k,m", [(90, 200, 75), (700, 96, 600), (4096, 40, 4096)])
@pytest.mark.parametrize("swap", [False, True])
def test_small_elements_beside_large_ones(n, k, m, small, large, swap):
    """Elements that bf16 alone has few bits for, in rows whose other elements
    are ordinary and meet zeros: each output keeps fp32's precision.  (In fp32
    the small ones are denormal from 2^-127 on: exact inputs, fewer bits.)"""
    a, b = _u((n, k), 14), _u((k, m), 15)
    a[:, ::2] *= np.float32(2.0 ** small)
    b[::2] = np.ldexp(b[::2], large)
    b[1::2, : m // 2] = 0
    b[1::2, m // 2:] *= np.float32(2.0 ** -40)
    if swap:
        a, b = np.ascontiguousarray(b.T), np.ascontiguousarray(a.T)
    rows = np.arange(0, a.shape[0], max(1, a.shape[0] // 64))
    ref = a[rows].astype(np.float64) @ b.astype(np.float64)
    assert (np.abs(G.gemm_ex(a, b)[rows] - ref) <= _bound(a[rows], b) + 2.0 ** -149 * k).all()


@pytest.mark.parametrize("ea,eb", [(-60, -60), (-70, -64), (-100, -40), (100, -100), (115, -120), (-130, 115), (60, 50)])
def test_magnitudes_of_operands(ea, eb):
    """Products that are small themselves, and operands of 2^111 and sums of
    2^96 and more, which the scaled split leaves to the fp32 instruction."""
    n, k, m = 130, 100, 90
    a, b = np.ldexp(_u((n, k), 16), ea), np.ldexp(_u((k, m), 17), eb)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    # Denormal results round at 2^-149, once per sum or part of it.
    assert (np.abs(G.gemm_ex(a, b) - ref) <= _bound(a, b) + 2.0 ** -149 * k).all()
