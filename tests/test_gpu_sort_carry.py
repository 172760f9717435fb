"""The radix sort past 2048 tiles (8,388,608 keys), where the scan of a digit's
tile counts carries its running total into a second chunk, against a stable
sort."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8_388_608, 8_388_609, 17_000_001])
@pytest.mark.parametrize("kind", ["random", "few"])
def test_sort_pairs(native, n, kind):
    rng = np.random.default_rng(n)
    # few: every digit's total in three values, so the carry is large
    keys = rng.integers(0, 1 << 24, n, dtype=np.uint32) if kind == "random" else \
        np.array([0x010203, 0x010303, 0xFF0203], np.uint32)[rng.integers(0, 3, n)]
    print(f"[sort carry] n={n} {kind}", flush=True)
    vals = np.arange(n, dtype=np.uint32)
    bk, bv = native.DeviceBuffer.from_array(keys), native.DeviceBuffer.from_array(vals)
    scr = native.DeviceBuffer(native.lib().pppm_sort_scratch_bytes(n))
    native.check(native.lib().pppm_sort_pairs(bk.ptr, bv.ptr, C.c_uint32(n), C.c_uint32(24), scr.ptr, None))
    native.synchronize()
    order = np.argsort(keys, kind="stable").astype(np.uint32)
    np.testing.assert_array_equal(bk.to_array(np.uint32, n), keys[order])
    np.testing.assert_array_equal(bv.to_array(np.uint32, n), order)
