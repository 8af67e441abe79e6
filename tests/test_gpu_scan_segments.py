"""Prefix sums of more than one launch: arrays around one segment (2^28 - 2^20
elements) and of several, against torch's 64-bit sums on the device."""
import ctypes

import pytest

from back40computing_amd._lib import check, lib

pytestmark = pytest.mark.gpu

SEGMENT = (1 << 28) - (1 << 20)


@pytest.mark.parametrize("n", [SEGMENT, SEGMENT + 1, 2 * SEGMENT + 8193])
def test_scan_segments(n):
    import torch
    print("scan segments", n, flush=True)
    x = torch.randint(-2 ** 31, 2 ** 31, (n,), dtype=torch.int64, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    sums = torch.cumsum(x.bitwise_and_(0xFFFFFFFF), 0)
    x = x.to(torch.int32)
    torch.cuda.synchronize()
    total = ctypes.c_uint64()
    out = torch.empty_like(x)
    check(lib().b40c_scan_u32(x.data_ptr(), out.data_ptr(), n, 0, ctypes.byref(total)))
    assert total.value == int(sums[-1])
    assert torch.equal(out, sums.to(torch.int32))
    check(lib().b40c_scan_u32(x.data_ptr(), x.data_ptr(), n, 1, ctypes.byref(total)))
    assert total.value == int(sums[-1])
    assert int(x[0]) == 0 and torch.equal(x[1:], out[:-1])
