"""pppm_mg_smooth on a PPPM_F64 handle works on the caller's x and b alone, so
calls that share a handle may overlap: on grids of 128K cells and more, two
streams with their own x and b give what each gives by itself, and k iterations
in one call are bitwise k calls of one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _smooth(native, mg, x, b, iters, stream=None):
    native.check(native.lib().pppm_mg_smooth(mg.h, x.ptr, b.ptr, iters, native.C.c_double(1.15), 0, stream))


@pytest.mark.parametrize("dims", [(64, 64, 64), (58, 57, 40), (128, 64, 48)])
def test_iterations_in_one_call_or_several(native, dims):
    n = int(np.prod(dims))
    rng = np.random.default_rng(sum(dims))
    x0, b = rng.standard_normal(n), native.DeviceBuffer.from_array(rng.standard_normal(n))
    mg = native.MG(dims, native.F64)
    one, many = native.DeviceBuffer.from_array(x0), native.DeviceBuffer.from_array(x0)
    print(f"[mg handle] dims={dims}", flush=True)
    _smooth(native, mg, one, b, 5)
    for _ in range(5):
        _smooth(native, mg, many, b, 1)
    native.synchronize()
    np.testing.assert_array_equal(one.to_array(np.float64, n), many.to_array(np.float64, n))


def test_two_streams_share_a_handle(native):
    dims, n = (128, 128, 128), 128 ** 3
    rng = np.random.default_rng(3)
    mg = native.MG(dims, native.F64)
    owners = [native.Context(native.config_params(8)) for _ in range(2)]  # each with a stream of its own
    streams = [c.stream for c in owners]
    xs = [rng.standard_normal(n) for _ in streams]
    bs = [native.DeviceBuffer.from_array(rng.standard_normal(n)) for _ in streams]
    alone = [native.DeviceBuffer.from_array(x) for x in xs]
    for x, b in zip(alone, bs):
        print("[mg handle] alone", flush=True)
        _smooth(native, mg, x, b, 8)
        native.synchronize()
    both = [native.DeviceBuffer.from_array(x) for x in xs]
    native.synchronize()
    print("[mg handle] overlapping", flush=True)
    for x, b, st in zip(both, bs, streams):
        _smooth(native, mg, x, b, 8, st)
    native.synchronize()
    for x, y in zip(both, alone):
        np.testing.assert_array_equal(x.to_array(np.float64, n), y.to_array(np.float64, n))
