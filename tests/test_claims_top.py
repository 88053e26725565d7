"""Claims at the top of the 32-bit index range: shares whose end is the greatest
index, on the host, and on the GPU programs over the last starts below 2^32 - 1,
each of which runs once, and none below them."""

import ctypes

import numpy as np
import pytest

import oracle_lib as O

TOP = (1 << 32) - 1


def steps(first, limit, n):
    f = O.lib().oracle_share_steps
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_uint32] * 3 + [ctypes.c_void_p]
    marks = np.zeros(max(1, limit - first), np.uint32)
    outside = f(first, limit, n, marks.ctypes.data)
    return outside, marks[:max(0, limit - first)]


@pytest.mark.parametrize("size", [0, 1, 30, 63, 64, 65, 200, 2048])
@pytest.mark.parametrize("limit", [2048, 0x80000000, 0xF0000001, TOP])
@pytest.mark.parametrize("n", [1, 37, 64])
def test_shares_cover_their_range_once(size, limit, n):
    outside, marks = steps(limit - size, limit, n)
    assert outside == 0 and (marks == 1).all()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,size,cycles", [("async", 1 << 14, 1 << 20), ("event", 1 << 20, 4)])
@pytest.mark.parametrize("count,groups", [(1, 1), (100, 3), (70001, 256)])
def test_last_starts(kind, size, cycles, count, groups):
    import harmonize_amd as hz

    first = TOP - count
    low = 1 << 20
    out = hz.DeviceArray(TOP, np.uint32)  # a count for every index, so that none is written out of range
    untouched = np.full(low, 0xABCD, np.uint32)
    hz.lib().harmonize_memcpy_host_to_device(out.ptr, untouched.ctypes.data, untouched.nbytes)
    it = hz.DeviceArray.from_numpy(np.array([first, TOP], np.uint32))
    inst = hz.Instance(kind, hz.SPEC_COLLATZ, size, hz.CollatzState(None, out.ptr, it.ptr))
    try:
        inst.init(groups)
        for _ in range(2000):
            inst.exec(groups, cycles)
            if inst.complete():
                break
        else:
            raise AssertionError("the program did not complete")
        got = np.empty(count, np.uint32)
        hz.lib().harmonize_memcpy_device_to_host(got.ctypes.data, out.ptr + 4 * first, got.nbytes)
        want, _ = O.collatz_steps(np.arange(first, TOP, dtype=np.uint64))
        assert np.array_equal(got, want)
        back = np.empty(low, np.uint32)
        hz.lib().harmonize_memcpy_device_to_host(back.ctypes.data, out.ptr, back.nbytes)
        assert np.array_equal(back, untouched)
        assert it.numpy()[0] >= TOP
    finally:
        inst.close()
