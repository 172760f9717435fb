"""Results do not depend on which kernel a level takes.  Levels are given to
tile passes, passes of two iterations, the small levels' one launch or launches
per half-sweep by their size, the number of components and a switch; all of them
do the same arithmetic, so the results are compared bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cycles(native, dims, dtype, b, x0, nu, sched, omega, small=True):
    """x after two V-cycles or one full-multigrid solve, all components."""
    ncomp = b.shape[0]
    mg = native.MG(dims, dtype, ncomp=ncomp)
    mg.set_small_levels(small)
    bx, bb = native.DeviceBuffer.from_array(x0), native.DeviceBuffer.from_array(b)
    if sched == "fmg":
        mg.solve(bx.ptr, bb.ptr, native.MG_REF_FMG, nu[0], nu[1], omega, 0.0, 1)
    else:
        mg.vcycles(bx.ptr, bb.ptr, 2, nu[0], nu[1], omega)
    native.synchronize()
    return bx.to_array(b.dtype, b.size).reshape(b.shape)


@pytest.mark.parametrize("dims,ncomp,dtype,nu,sched",
                         [((40, 40, 40), 4, 2, (4, 4), "fmg"),      # one component in tiles, four past 128K cells
                          ((65, 65, 65), 12, 2, (4, 4), "fmg"),     # odd: no pass of two iterations
                          ((50, 36, 44), 6, 2, (2, 3), "vcycle"),   # a ghost factor on the coarse levels
                          ((33, 35, 31), 7, 2, (2, 2), "vcycle"),   # odd levels
                          ((64, 64, 64), 3, 1, (2, 2), "vcycle"),   # tiles of 8^3 alone, of 16^3 together
                          ((50, 68, 62), 4, 1, (2, 1), "vcycle"),   # ... that the grid does not fill
                          ((64, 64, 64), 4, 1, (2, 1), "vcycle"),   # together in blocked passes
                          ((66, 64, 68), 3, 1, (1, 2), "vcycle"),
                          ((34, 34, 34), 12, 1, (1, 1), "vcycle"),  # ... as they fill their tiles badly
                          ((64, 64, 2), 12, 1, (2, 2), "vcycle"),   # thin: half-sweeps together
                          ((38, 54, 141), 3, 1, (2, 2), "vcycle"),  # odd nz: smoothing alone out of place
                          ((65, 66, 68), 16, 1, (2, 1), "vcycle"),  # odd nx
                          ((32, 32, 32), 48, 1, (2, 2), "vcycle")])
def test_component_equals_alone(native, dims, ncomp, dtype, nu, sched):
    t = np.float64 if dtype == native.F64 else np.float32
    rng = np.random.default_rng(sum(dims))
    shape = (ncomp, int(np.prod(dims)))
    b, x0 = rng.standard_normal(shape).astype(t), rng.standard_normal(shape).astype(t)
    print(f"[mg choice] dims={dims} ncomp={ncomp} {t.__name__} nu={nu} {sched}", flush=True)
    both = _cycles(native, dims, dtype, b, x0, nu, sched, 1.15)
    assert np.all(np.isfinite(both))
    for c in {0, ncomp // 2, ncomp - 1}:
        alone = _cycles(native, dims, dtype, b[c:c + 1], x0[c:c + 1], nu, sched, 1.15)
        np.testing.assert_array_equal(both[c], alone[0])


@pytest.mark.parametrize("dims,nu", [((64, 64, 64), (2, 2)), ((64, 64, 64), (1, 1)), ((96, 72, 80), (2, 1)),
                                     ((80, 112, 72), (1, 2)), ((128, 64, 64), (2, 2)),
                                     ((62, 58, 60), (2, 2)), ((62, 58, 60), (2, 1)),  # partial tiles of 16^3
                                     ((46, 62, 30), (2, 2))])                         # ... and of 8^3
def test_blocked_kinds_equal_half_sweeps(native, dims, nu):
    """FP32 V-cycles of one launch per half-sweep and in blocked passes (kinds 1
    to 4) and tiles, three components."""
    rng = np.random.default_rng(sum(dims))
    shape = (3, int(np.prod(dims)))
    b, x0 = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(shape).astype(np.float32)
    out = []
    for kind in (0, 1, 2, 3, 4):
        print(f"[mg choice] dims={dims} nu={nu} kind={kind}", flush=True)
        mg = native.MG(dims, native.F32, ncomp=3)
        mg.set_blocked(kind)
        if kind == 3:
            mg.set_blocked_min_cells(1)  # every level above the coarsest two
        bx, bb = native.DeviceBuffer.from_array(x0), native.DeviceBuffer.from_array(b)
        mg.vcycles(bx.ptr, bb.ptr, 2, nu[0], nu[1], 1.15)
        native.synchronize()
        out.append(bx.to_array(np.float32, b.size))
    for o in out[1:]:
        np.testing.assert_array_equal(o, out[0])


@pytest.mark.parametrize("dims", [(16, 16, 16), (12, 20, 14), (2, 160, 14), (22, 22, 22), (32, 32, 32), (5, 139, 57),
                                  (1, 6, 300)])
def test_small_levels_switch_without_the_one_launch(native, dims):
    """pppm_mg_set_small_levels changes no bit where the one launch does not
    apply either: two levels (16^3 above 8^3), or one it cannot hold."""
    rng = np.random.default_rng(sum(dims))
    shape = (2, int(np.prod(dims)))
    b, x0 = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(shape).astype(np.float32)
    print(f"[mg choice] switch dims={dims}", flush=True)
    on, off = (_cycles(native, dims, native.F32, b, x0, (2, 2), "vcycle", 1.15, small) for small in (True, False))
    np.testing.assert_array_equal(on, off)


@pytest.mark.parametrize("dims", [(64, 64, 64), (32, 32, 32), (96, 80, 72)])
def test_gauss_seidel_forgets_what_it_replaces(native, dims):
    """omega = 1 in FP64: the first half-sweep replaces every odd cell by a value
    that does not hold the old one, however large that was."""
    nx, ny, nz = dims
    rng = np.random.default_rng(7)
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    odd = ((i + j + k) & 1).ravel() == 1
    b = rng.standard_normal((1, odd.size))
    x0 = rng.standard_normal((1, odd.size))
    x1 = np.where(odd, 1e12 * rng.standard_normal(odd.size), x0[0])[None]
    print(f"[mg choice] omega=1 dims={dims}", flush=True)
    np.testing.assert_array_equal(_cycles(native, dims, native.F64, b, x0, (2, 2), "vcycle", 1.0),
                                  _cycles(native, dims, native.F64, b, x1, (2, 2), "vcycle", 1.0))
