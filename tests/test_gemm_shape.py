"""How a product is cut (ember_amd/csrc/gemm_shape.h) at extents up to
2^31 - 1, where a sum of an extent and a tile passes the largest int."""

import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ember_amd", "csrc")
TOP = 2 ** 31 - 1
SOURCE = """
#include "gemm_shape.h"
extern "C" void choose(int64_t n, int64_t m, int64_t k, int64_t batch, int64_t *out)
{
    const ember::GemmChoice c = ember::choose_gemm(n, m, k, batch, 256);
    out[0] = c.shape, out[1] = c.ksplit, out[2] = c.kchunk;
}
extern "C" void range(int k, int chunk, int z, int slab, int64_t *out)
{
    const ember::KRange r = ember::k_range(k, chunk, z, slab);
    out[0] = r.beg, out[1] = r.end, out[2] = r.slabs, out[3] = r.first;
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("gemm_shape")
    (d / "s.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ftrapv", "-fPIC", "-shared", "-I", CSRC, "s.cpp", "-o", "s.so"], cwd=d, check=True)
    L = C.CDLL(str(d / "s.so"))
    L.choose.argtypes = [C.c_int64] * 4 + [C.c_void_p]

    def call(f, *args):
        out = (C.c_int64 * 4)()
        f(*args, out)
        return list(out)
    return lambda *a: call(L.choose, *a)[:3], lambda *a: call(L.range, *a)


@pytest.mark.parametrize("k", [1, 63, 64, 4096, 2 ** 30, 1431655764, 1431655765, 1500000000, 2000000000, 2147483600, TOP])
@pytest.mark.parametrize("n,m", [(1, 1), (300, 1), (1, 513), (64, 64), (4096, 4096)])
def test_splits_cover_k(shape, n, m, k):
    choose, k_range = shape
    tile, splits, chunk = choose(n, m, k, 1)
    assert 0 <= tile < 3 and 1 <= splits <= 64 and 1 <= chunk <= k + 31
    for slab in (16, 32):
        at = 0
        for z in range(splits):
            beg, end, slabs, first = k_range(k, chunk, z, slab)
            assert beg == at < end and 1 <= first <= slab and first + (slabs - 1) * slab == end - beg
            at = end
        assert at == k


@pytest.mark.parametrize("n,m", [(TOP, 1), (1, TOP), (2 ** 30 + 1, 1), (1100000000, 30), (TOP - 255, 2)])
@pytest.mark.parametrize("k", [0, 1, 40])
def test_long_outputs(shape, n, m, k):
    choose, k_range = shape
    assert choose(n, m, k, 1)[1] == 1
    assert k_range(k, k, 0, 32)[:3] == [0, k, (k + 31) // 32]
