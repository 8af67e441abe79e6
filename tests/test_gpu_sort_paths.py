"""The radix sort at the sizes where its form changes: the one-workgroup limit,
tile and block edges, every policy, places whose keys share a digit, the fixed
scratch that makes blocks grow, and 64-bit look-back words.  Results are
compared bit for bit with numpy's stable sort of the ordered key bits, the
selector with the number of places that move keys."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TYPES = [np.uint32, np.int32, np.float32, np.uint64, np.int64, np.float64]
SIZES = [2, 63, 64, 65, 1024, 8191, 8192, 8193, 12287, 12288, 12289, 70_001, 4_194_304 + 4097]


def _ordered(keys):
    """The unsigned view whose order is the sort's."""
    bits = keys.view(np.uint32 if keys.dtype.itemsize == 4 else np.uint64)
    high = bits.dtype.type(1) << bits.dtype.type(8 * keys.dtype.itemsize - 1)
    if keys.dtype.kind == "i":
        return bits ^ high
    if keys.dtype.kind == "f":
        return np.where(bits & high, ~bits, bits ^ high)
    return bits


def _expect(keys, begin, end):
    o = _ordered(keys)
    width = end - begin
    part = o >> o.dtype.type(begin)
    if width < 8 * o.dtype.itemsize:
        part &= (o.dtype.type(1) << o.dtype.type(width)) - o.dtype.type(1)
    places = 0
    for s in range(0, width, 8):
        d = (part >> part.dtype.type(s)) & part.dtype.type(255)
        places += int(d.min() != d.max())
    return np.argsort(part, kind="stable"), places & 1


def _keys(dtype, n, seed):
    rng = np.random.default_rng(seed)
    bits = rng.integers(0, 1 << 63, n, dtype=np.uint64) * 2 + rng.integers(0, 2, n, dtype=np.uint64)
    k = bits.astype(np.uint32).view(dtype) if np.dtype(dtype).itemsize == 4 else bits.view(dtype)
    if np.dtype(dtype).kind == "f":
        k = np.where(np.isnan(k), np.dtype(dtype).type(-1.5), k)
    k[rng.integers(0, n, n // 3)] = k[0]
    return k


def _check(keys, with_values, begin=0, end=None, policy=(0, 0)):
    from back40computing_amd import radix_sort as rs
    end = 8 * keys.dtype.itemsize if end is None else end
    db = rs.DoubleBuffer(keys.dtype, keys.size, with_values=with_values)
    db.d_keys[0].upload(keys)
    if with_values:
        db.d_values[0].upload(np.arange(keys.size, dtype=np.uint32))
    en = rs.Enactor()
    en.set_policy(*policy)
    assert en.Sort(db, keys.size, begin, end) == 0
    order, parity = _expect(keys, begin, end)
    assert db.selector == parity
    word = np.uint32 if keys.dtype.itemsize == 4 else np.uint64
    got = db.d_keys[db.selector].download(word, keys.size)
    np.testing.assert_array_equal(got, keys.view(word)[order])
    if with_values:
        np.testing.assert_array_equal(db.d_values[db.selector].download(np.uint32, keys.size), order)
    en.close()


@pytest.mark.parametrize("dtype", TYPES, ids=[np.dtype(t).name for t in TYPES])
@pytest.mark.parametrize("with_values", [False, True], ids=["keys", "pairs"])
def test_sizes(dtype, with_values):
    for n in SIZES:
        print("sort", np.dtype(dtype).name, with_values, n, flush=True)
        _check(_keys(dtype, n, n), with_values)


@pytest.mark.parametrize("n", [5000, 20_000, 300_000])
def test_bit_ranges_and_shared_digits(n):
    rng = np.random.default_rng(n)
    for begin, end in ((0, 1), (3, 10), (5, 44), (8, 64), (63, 64), (0, 57)):
        print("bits", n, begin, end, flush=True)
        _check(_keys(np.uint64, n, end), True, begin, end)
    same = np.full(n, 0x1234567890ABCDEF, np.uint64)
    _check(same, True)
    same[1:] = (same[1:] & ~np.uint64(0xFF0000)) | (rng.integers(0, 256, n - 1).astype(np.uint64) << np.uint64(16))
    _check(same, True)
    _check(np.sort(_keys(np.int64, n, 1)), False)


@pytest.mark.parametrize("policy", [(8, 1), (16, 0), (16, 1), (8, 8), (0, 3)])
def test_policies(policy):
    for n in (8193, 1_000_003, 9_000_000):
        print("policy", policy, n, flush=True)
        _check(_keys(np.uint32, n, n), True, policy=policy)
        _check(_keys(np.uint64, n, n), False, 0, 24, policy=policy)


def test_fixed_scratch_grows_blocks():
    from back40computing_amd import _lib, radix_sort as rs
    lib = _lib.lib()
    n = 21_000_001
    keys = _keys(np.uint64, n, 9)
    a, b = rs.DeviceArray(keys.nbytes), rs.DeviceArray(keys.nbytes)
    a.upload(keys)
    sel = ctypes.c_int32()
    assert lib.b40c_radix_sort_u64_noalloc(a.ptr, b.ptr, n, 0, 64, ctypes.byref(sel)) == 0
    np.testing.assert_array_equal((b if sel.value else a).download(np.uint64, n), np.sort(keys))


def test_wide_look_back_words():
    """2^30 keys and more: counts no longer fit 30 bits.  Keys hold their
    index above an 8-bit digit, so the sorted order is checked as one strictly
    increasing sequence."""
    from back40computing_amd import _lib, radix_sort as rs
    lib = _lib.lib()
    n, step = (1 << 30) + 12345, 1 << 27
    a, b = rs.DeviceArray(8 * n), rs.DeviceArray(8 * n)
    for i in range(0, n, step):
        index = np.arange(i, min(n, i + step), dtype=np.uint64)
        digit = (index * np.uint64(2654435761) >> np.uint64(13)) & np.uint64(255)
        digit[index < n // 2] = 7
        keys = (index << np.uint64(8)) | digit
        assert lib.b40c_memcpy_h2d(ctypes.c_void_p(a.ptr.value + 8 * i), ctypes.c_void_p(keys.ctypes.data), keys.nbytes) == 0
    sel = ctypes.c_int32()
    assert lib.b40c_radix_sort(rs.KEY_TYPES[np.dtype(np.uint64)], a.ptr, b.ptr, None, None, n, 0, 8,
                               ctypes.byref(sel)) == 0
    assert sel.value == 1
    total, last = 0, -1
    for i in range(0, n, step):
        keys = np.empty(min(step, n - i), np.uint64)
        assert lib.b40c_memcpy_d2h(ctypes.c_void_p(keys.ctypes.data), ctypes.c_void_p(b.ptr.value + 8 * i), keys.nbytes) == 0
        seq = ((keys & np.uint64(255)) << np.uint64(48)) | (keys >> np.uint64(8))
        assert bool((seq[1:] > seq[:-1]).all()) and int(seq[0]) > last, i
        last = int(seq[-1])
        total += int((keys >> np.uint64(8)).sum())
    assert total == n * (n - 1) // 2


def test_concurrent_enactors():
    errors = []

    def work(seed):
        try:
            for n in (6000, 300_000, 2_000_000):
                _check(_keys(np.uint64, n + seed, seed), True)
        except Exception as e:  # reported below, in the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


# Tiles of 4,096 keys around an XCD group (64), a serving step (256 and 128), the
# change of the step (512), and the keys from which tiles hold 8,192 on.
@pytest.mark.parametrize("n", [64 * 4096, 64 * 4096 + 1, 128 * 4096 + 1, 256 * 4096 + 1, 512 * 4096, 512 * 4096 + 1,
                               3_670_015, 3_670_016])
@pytest.mark.parametrize("dtype,values", [(np.uint32, True), (np.uint64, False), (np.float64, True)])
def test_chained_tiles(dtype, values, n):
    _check(_keys(dtype, n, n % 1000), values)
