"""Prefix sum and consecutive removal where their blocks chain: sizes around one
block (8,192 elements, 4,096 keys) and around the 256 blocks that one step of
the chain takes, in place and not, aligned and not."""
import ctypes

import numpy as np
import pytest

from back40computing_amd._lib import check, lib
from back40computing_amd.radix_sort import DeviceArray

pytestmark = pytest.mark.gpu

B = 8192
SCAN_SIZES = [1, 63, B - 1, B, B + 1, 2 * B + 5, 255 * B, 256 * B, 256 * B + 1, 600 * B - 3]
T = 4096
TRIM_SIZES = [1, 64, 65, T - 1, T, T + 1, 255 * T + 7, 256 * T, 257 * T + 1, 1100 * T - 63]


@pytest.mark.parametrize("n", SCAN_SIZES)
@pytest.mark.parametrize("exclusive", [1, 0])
@pytest.mark.parametrize("offset,in_place", [(0, False), (0, True), (4, True)])
def test_scan_blocks(n, exclusive, offset, in_place):
    x = np.random.default_rng(n + exclusive).integers(0, 1 << 32, n, dtype=np.uint32)
    src, dst = DeviceArray(4 * n + 16), DeviceArray(4 * n + 16)
    check(lib().b40c_memcpy_h2d(src.ptr.value + offset, x.ctypes.data, x.nbytes))
    out = (src if in_place else dst).ptr.value + offset
    total = ctypes.c_uint64()
    check(lib().b40c_scan_u32(src.ptr.value + offset, out, n, exclusive, ctypes.byref(total)))
    got = np.empty(n, np.uint32)
    check(lib().b40c_memcpy_d2h(got.ctypes.data, out, got.nbytes))
    wide = np.cumsum(x, dtype=np.uint64)
    assert total.value == int(wide[-1])
    want = wide - x if exclusive else wide
    assert np.array_equal(got, want.astype(np.uint32))


@pytest.mark.parametrize("n", TRIM_SIZES)
@pytest.mark.parametrize("distinct", ["few", "half", "all", "one"])
@pytest.mark.parametrize("values,offset", [(True, 0), (False, 0), (True, 1)])
def test_trim_blocks(n, distinct, values, offset):
    rng = np.random.default_rng(n)
    step = {"few": rng.random(n) < 1e-3, "half": rng.random(n) < 0.5,
            "all": np.ones(n, bool), "one": np.zeros(n, bool)}[distinct]
    # keys with a zero first run, so the padding value of a block is a key too
    keys = np.cumsum(step).astype(np.uint64) * np.uint64(0x100000001)
    keys -= keys[0]
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint32)
    head = np.concatenate(([True], keys[1:] != keys[:-1]))
    m = int(head.sum())
    ki, vi = DeviceArray(8 * n + 16), DeviceArray(4 * n + 16)
    ko, vo = DeviceArray(8 * n + 16), DeviceArray(4 * n + 16)
    guard = np.full(n + 2, 0xDEADBEEF, np.uint64)
    ko.upload(guard)
    k_at, v_at = ki.ptr.value + 8 * offset, vi.ptr.value + 4 * offset
    check(lib().b40c_memcpy_h2d(k_at, keys.ctypes.data, keys.nbytes))
    check(lib().b40c_memcpy_h2d(v_at, vals.ctypes.data, vals.nbytes))
    count = ctypes.c_int64()
    check(lib().b40c_consecutive_removal_u64(k_at, v_at if values else None, ko.ptr, vo.ptr if values else None, n,
                                             ctypes.byref(count)))
    assert count.value == m
    got = ko.download(np.uint64, n + 2)
    assert np.array_equal(got[:m], keys[head])
    assert np.array_equal(got[m:], guard[m:])
    if values:
        assert np.array_equal(vo.download(np.uint32, m), vals[head])
