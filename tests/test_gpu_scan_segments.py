"""Prefix sums of more than one launch: arrays around one segment (2^28 - 2^20
elements) and of several, exclusive and, in place, inclusive."""
import ctypes

import numpy as np
import pytest

from back40computing_amd._lib import check, lib
from back40computing_amd.radix_sort import DeviceArray

pytestmark = pytest.mark.gpu

SEGMENT = (1 << 28) - (1 << 20)


@pytest.mark.parametrize("n", [SEGMENT, SEGMENT + 1, 2 * SEGMENT + 8193])
def test_scan_segments(n):
    print("scan segments", n, flush=True)
    x = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint32)
    incl = np.cumsum(x, dtype=np.uint32)  # modulo 2^32
    sum64 = int(x.sum(dtype=np.uint64))
    src, dst = DeviceArray(4 * n), DeviceArray(4 * n)
    src.upload(x)
    total = ctypes.c_uint64()
    check(lib().b40c_scan_u32(src.ptr, dst.ptr, n, 1, ctypes.byref(total)))
    assert total.value == sum64
    out = dst.download(np.uint32, n)
    assert out[0] == 0 and np.array_equal(out[1:], incl[:-1])
    check(lib().b40c_scan_u32(src.ptr, src.ptr, n, 0, ctypes.byref(total)))
    assert total.value == sum64
    assert np.array_equal(src.download(np.uint32, n), incl)
