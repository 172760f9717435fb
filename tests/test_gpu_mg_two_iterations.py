"""The blocked pass of two red-black iterations (64 x 64 cell regions marching
in z, tiles of 56 or 52 cells) against one launch per half-sweep: dimensions
one pair or row off a tile, smaller than a halo, one plane, z chunks that end
unevenly, odd ny and nz, and each pass of a V-cycle (from zero, from an
iterate with the residual's wider halo, with the prolongation)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(56, 56, 8), (58, 57, 9), (54, 55, 130), (2, 3, 5), (114, 1, 7), (64, 113, 1),
                                  (170, 52, 33)])
@pytest.mark.parametrize("iters", [2, 5])
def test_smooth_equals_halfsweeps(native, dims, iters):
    """Ten half-sweeps add about ten roundings of 6e-8 of the largest value
    in each cell."""
    n = int(np.prod(dims))
    rng = np.random.default_rng(sum(dims))
    x0, b = rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    out = []
    for kind in (0, 4):
        print(f"[mg two] smooth dims={dims} iters={iters} kind={kind}", flush=True)
        mg = native.MG(dims, native.F32)
        bx, bb = native.DeviceBuffer.from_array(x0), native.DeviceBuffer.from_array(b)
        native.check(native.lib().pppm_mg_smooth(mg.h, bx.ptr, bb.ptr, iters, native.C.c_double(1.15), kind, None))
        native.synchronize()
        out.append(bx.to_array(np.float32, n))
    assert np.max(np.abs(out[1] - out[0])) <= 1e-5 * np.max(np.abs(out[0]))


@pytest.mark.parametrize("dims,ncomp,nu", [((112, 56, 64), 1, (2, 2)), ((114, 60, 50), 2, (2, 2)), ((52, 104, 28), 3, (2, 2)),
                                           ((160, 54, 58), 1, (2, 1)), ((72, 72, 72), 1, (1, 2)), ((150, 150, 150), 1, (2, 2))])
def test_vcycles_equal_halfsweeps(native, dims, ncomp, nu):
    """Every level of even dimensions in blocked passes (150^3: the odd
    second level per half-sweep), from a zero start and from the iterate."""
    n = ncomp * int(np.prod(dims))
    b = np.random.default_rng(sum(dims)).standard_normal(n).astype(np.float32)
    out = []
    for kind in (0, 4):
        print(f"[mg two] vcycles dims={dims} ncomp={ncomp} nu={nu} kind={kind}", flush=True)
        mg = native.MG(dims, native.F32, ncomp=ncomp)
        mg.set_blocked(kind)
        if dims[0] != 150:
            mg.set_blocked_min_cells(1)
        bx, bb = native.DeviceBuffer(4 * n), native.DeviceBuffer.from_array(b)
        bx.fill_zero()
        mg.vcycles(bx.ptr, bb.ptr, 1, nu[0], nu[1], 1.15, x_zero=True)
        mg.vcycles(bx.ptr, bb.ptr, 2, nu[0], nu[1], 1.15)
        native.synchronize()
        out.append(bx.to_array(np.float32, n))
    assert np.all(np.isfinite(out[1]))
    assert rel_l2(out[1], out[0]) < 1e-5


@pytest.mark.parametrize("dims,nu", [((96, 80, 72), (4, 4)), ((114, 73, 66), (3, 2)), ((112, 96, 49), (2, 5))])
def test_full_multigrid_fp64_large_level(native, oracle, dims, nu):
    """One full-multigrid pass in FP64 whose finest level takes the pass of
    two iterations (56 x 24 tiles): the oracle's iterate to 1e-10."""
    n = int(np.prod(dims))
    b = np.random.default_rng(sum(dims)).standard_normal(n)
    omega = float(np.float32(1.43))
    mg = native.MG(dims, native.F64)
    bx, bb = native.DeviceBuffer(8 * n), native.DeviceBuffer.from_array(b)
    bx.fill_zero()
    print(f"[mg two] FMG dims={dims} nu={nu}", flush=True)
    mg.solve(bx.ptr, bb.ptr, native.MG_REF_FMG, nu[0], nu[1], omega, 0.0, 1)
    x = bx.to_array(np.float64, n)
    xo, _, _ = oracle.mg_solve(b, dims, schedule=oracle.MG_REF_FMG, nu1=nu[0], nu2=nu[1], omega=omega)
    assert rel_l2(x, xo) < 1e-10
