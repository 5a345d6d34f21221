"""The INT8 GEMM's host mirror (csrc/capi.hip): int32 lists packed into one
buffer up to 1 MB, and above that into a staging buffer of two 256 KB halves.
Sizes around both and around the 16 codes that one packing step takes; codes at
and past the int8 range at the first, middle and last place; a refused call
followed by a good one on the same context."""
import ctypes as C

import numpy as np
import pytest

from tokenvector.inference_amd import _lib

pytestmark = pytest.mark.gpu

# one code; K below, at and past 16; packed bytes of exactly 1 MB (1024 x 1024)
# and of one row more (the first that goes through the halves); rows split over
# halves (11 rows of K = 100 000); many halves
SHAPES = [(1, 1, 1), (3, 5, 15), (2, 7, 17), (256, 256, 1024), (257, 256, 1023), (1, 65537, 16),
          (300, 1000, 131), (5, 9, 100000), (1030, 2304, 768), (1024, 3, 1024), (1025, 512, 1024),
          (3, 1025, 1020), (5, 11, 100000)]


def _accum(a, w, m, n, k):
    acc = np.full(m * n, 7, np.int32)
    p = [v.ctypes.data_as(C.c_void_p) for v in (a, w, acc)]
    rc = _lib.lib().tkv_hip_matmul_int8_accum(*p, m, n, k)
    return rc, acc.reshape(m, n)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_host_gemm_staging(hip, m, n, k):
    print(f"host staging {m}x{n}x{k}", flush=True)
    r = np.random.default_rng(m * 31 + n + k)
    a = r.integers(-128, 128, m * k).astype(np.int32)
    w = r.integers(-128, 128, n * k).astype(np.int32)
    want = a.reshape(m, k).astype(np.float64) @ w.reshape(n, k).astype(np.float64).T  # exact
    for _ in range(2):
        rc, acc = _accum(a, w, m, n, k)
        assert rc == _lib.OK
        assert np.array_equal(acc.astype(np.float64), want)
    for at in (0, n * k // 2, n * k - 1):
        for code in (128, -129, 2**31 - 1, -2**31):
            bad = w.copy()
            bad[at] = code
            assert _accum(a, bad, m, n, k)[0] == _lib.UNSUPPORTED, (at, code)
    rc, acc = _accum(a, w, m, n, k)
    assert rc == _lib.OK
    assert np.array_equal(acc.astype(np.float64), want)
