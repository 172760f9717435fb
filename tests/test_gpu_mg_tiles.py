"""Multigrid levels that take the tile passes (3-D tiles in LDS, up to two
red-black iterations a launch) against the oracle and against one launch per
half-sweep: dimensions that leave partial tiles, tiles with a halo on every
side, one level only, odd coarse levels and odd iteration counts."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,nu", [((16, 16, 16), (4, 4)), ((50, 36, 44), (4, 4)), ((64, 18, 34), (3, 2)),
                                     ((40, 40, 40), (2, 3)), ((80, 64, 48), (4, 4)), ((17, 15, 19), (4, 1))])
def test_full_multigrid_fp64_against_oracle(native, oracle, dims, nu):
    """One full-multigrid pass of the reference's schedule, FP64: the
    oracle's iterate to 1e-10."""
    n = int(np.prod(dims))
    b = np.random.default_rng(sum(dims)).standard_normal(n)
    omega = float(np.float32(1.43))
    mg = native.MG(dims, native.F64)
    bx, bb = native.DeviceBuffer(8 * n), native.DeviceBuffer.from_array(b)
    bx.fill_zero()
    print(f"[mg tiles] FMG dims={dims} nu={nu}", flush=True)
    mg.solve(bx.ptr, bb.ptr, native.MG_REF_FMG, nu[0], nu[1], omega, 0.0, 1)
    x = bx.to_array(np.float64, n)
    xo, _, _ = oracle.mg_solve(b, dims, schedule=oracle.MG_REF_FMG, nu1=nu[0], nu2=nu[1], omega=omega)
    assert rel_l2(x, xo) < 1e-10


@pytest.mark.parametrize("dims,ncomp,nu", [((24, 40, 18), 1, (2, 2)), ((96, 96, 96), 3, (2, 2)), ((66, 34, 130), 1, (1, 2)),
                                           ((100, 100, 100), 1, (2, 1)), ((64, 64, 64), 3, (1, 1))])
def test_vcycle_fp32_tiles_equal_halfsweeps(native, dims, ncomp, nu):
    """FP32 V-cycles with tile passes equal the launch-per-half-sweep ones to
    rounding, from a zero start and from the previous iterate."""
    n = ncomp * int(np.prod(dims))
    b = np.random.default_rng(sum(dims)).standard_normal(n).astype(np.float32)
    out = []
    for kind in (0, 2):
        print(f"[mg tiles] vcycles dims={dims} ncomp={ncomp} nu={nu} kind={kind}", flush=True)
        mg = native.MG(dims, native.F32, ncomp=ncomp)
        mg.set_blocked(kind)
        bx, bb = native.DeviceBuffer(4 * n), native.DeviceBuffer.from_array(b)
        bx.fill_zero()
        mg.vcycles(bx.ptr, bb.ptr, 1, nu[0], nu[1], 1.15, x_zero=True)
        mg.vcycles(bx.ptr, bb.ptr, 2, nu[0], nu[1], 1.15)
        native.synchronize()
        out.append(bx.to_array(np.float32, n))
    assert np.all(np.isfinite(out[1]))
    assert rel_l2(out[1], out[0]) < 1e-5
