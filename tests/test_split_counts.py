"""The K split that kh_gemm plans (kh_gemm_split_count_for), which needs no device: an undivided card's 256
compute units are assumed before the backend is initialised."""
import ctypes as C

import pytest

from kandle_amd import _lib

BF16, F32 = 1, 0


def _count(m, n, k, dtype):
    out = C.c_int(-1)
    _lib.check(_lib.load().kh_gemm_split_count_for(m, n, k, dtype, C.byref(out)))
    return out.value


@pytest.mark.parametrize("m,n,k,dtype,count", [
    (512, 1024, 3072, F32, 4), (1000, 1024, 3072, BF16, 1), (256, 2560, 9728, BF16, 3), (9, 2560, 4096, F32, 8),
    (8, 1024, 3072, BF16, 8), (8, 1024, 3072, F32, 1), (8, 1024, 1024, BF16, 1), (512, 1024, 640, BF16, 1),
    (9, 0, 2048, BF16, 1), (0, 8, 2048, BF16, 1), (9, 8, 0, F32, 1), (9, 1024, 2044, BF16, 1)])
def test_counts(m, n, k, dtype, count):
    assert _count(m, n, k, dtype) == count


def test_parts_are_whole_and_cover_k():
    """At most eight parts of a multiple of 128 columns, none of them empty."""
    for m in (2, 8, 9, 33, 64, 200, 512, 1000, 2000):
        for n in (4, 64, 1000, 1024, 6144):
            for k in (512, 520, 1024, 2056, 4096, 9728):
                for dtype in (BF16, F32):
                    parts = _count(m, n, k, dtype)
                    width = -(-(-(-k // parts)) // 128) * 128
                    assert 1 <= parts <= 8 and (parts == 1 or -(-k // width) == parts), (m, n, k, dtype, parts)
