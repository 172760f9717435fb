"""The radix sort at the sizes where its tiles change (one key, tile edges of
1024, 2048 and 4096 keys, the lines at 2^19 and 3 * 2^19 keys between them), with constant and
descending keys, and a context's cell tables on both sides of the line between
searched and scanned offsets (101^3 and 102^3 cells)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 1 << 19, (1 << 19) + 1, 3 << 19, (3 << 19) + 1, 2_100_001])
@pytest.mark.parametrize("kind", ["random", "constant", "descending"])
def test_sort_pairs_sizes(native, n, kind):
    rng = np.random.default_rng(n)
    if kind == "random":
        keys = rng.integers(0, 1 << 21, n, dtype=np.uint32)
    else:
        keys = np.full(n, 0x12345, np.uint32) if kind == "constant" else np.arange(n, dtype=np.uint32)[::-1] >> 1
    vals = rng.permutation(n).astype(np.uint32)
    print(f"[sort] n={n} {kind}", flush=True)
    bk, bv = native.DeviceBuffer.from_array(keys), native.DeviceBuffer.from_array(vals)
    scr = native.DeviceBuffer(native.lib().pppm_sort_scratch_bytes(n))
    native.check(native.lib().pppm_sort_pairs(bk.ptr, bv.ptr, C.c_uint32(n), C.c_uint32(21), scr.ptr, None))
    native.synchronize()
    order = np.argsort(keys, kind="stable")
    np.testing.assert_array_equal(bk.to_array(np.uint32, n), keys[order])
    np.testing.assert_array_equal(bv.to_array(np.uint32, n), vals[order])


def test_scratch_serves_smaller_sorts(native):
    """Scratch for n is at least that of every smaller count."""
    sizes = [1, 1024, 1025, 4096, 1 << 19, (1 << 19) + 1, 3 << 19, (3 << 19) + 1, 4_194_304, 4_194_305, 1 << 24]
    need = [native.lib().pppm_sort_scratch_bytes(q) for q in sizes]
    assert need == sorted(need)


@pytest.mark.parametrize("g", [2, 101, 102])
@pytest.mark.parametrize("n", [1, 50_001])
def test_cell_tables(native, g, n):
    rng = np.random.default_rng(g)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = 0.4 + 0.1 * rng.random((n, 3))
    pos[n // 2:, :3] = 0.999  # the last cell, and empty ones between
    w = rng.standard_normal((3, n))
    print(f"[sort] cell tables g={g} n={n}", flush=True)
    ctx = native.Context(native.config_params(g))
    sc = native.Scene(pos, w)
    ctx.set_vortices(sc.n, sc.pos.ptr, sc.w_ptrs())
    native.synchronize()
    _, _, st, en = ctx.sorted_vortices()
    start, end = native.dev_to_array(st, np.uint32, g ** 3), native.dev_to_array(en, np.uint32, g ** 3)
    h = np.float32(1.0 / g)
    c = np.floor(pos[:, :3] / h).astype(np.int64)
    key = np.sort((c[:, 2] * g + c[:, 1]) * g + c[:, 0])
    cells = np.arange(g ** 3)
    lo, hi = np.searchsorted(key, cells), np.searchsorted(key, cells, side="right")
    empty = lo == hi
    np.testing.assert_array_equal(start, np.where(empty, 0xFFFFFFFF, lo).astype(np.uint32))
    np.testing.assert_array_equal(end, np.where(empty, 0xFFFFFFFF, hi).astype(np.uint32))
