"""The far-field buffer against 64 bits where the grid vorticity is smooth.

dir is odd, so the local correction and the diagonal term are sums of
differences of the vorticity over a few cells; FP32 sums that hold the
vorticity itself lose the ratio of the two.  One vortex per cell centre gives
the grid exactly the field asked for, and the buffer is compared with the
formula in float64 on the grids that the context holds (psi and vorticity), so
only the correction's own rounding and the rounding of the stored float are
left.  The bound: 4 roundings of 2^-24 of the sum of |dir| h^3 times the
differences from the cell itself (each difference, each product, each partial
sum, each fold over an axis: their errors add as a random walk well inside the
sum of absolute values), the diagonal term alike, and half an ulp of the stored
float."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FOUR_PI, DIAG = 12.5663706144, 0.250580605913965
F32EPS = 2.0 ** -24


def _field(kind, g):
    z, y, x = np.meshgrid(*[(np.arange(g) + 0.5) / g] * 3, indexing="ij")
    if kind == "ripple":
        return [1 + 0.02 * np.sin(2 * np.pi * (x * (2 + q) + y * (3 - q) + z) + q) for q in range(3)]
    return [np.sin(np.pi * x + 0.3 * q) * np.sin(np.pi * y) * np.cos(np.pi * z) for q in range(3)]


def _clamped(f, ax):
    i = np.arange(f.shape[ax])
    return np.take(f, np.minimum(i + 1, i[-1]), ax), np.take(f, np.maximum(i - 1, 0), ax)


@pytest.mark.parametrize("kind", ["ripple", "low"])
@pytest.mark.parametrize("g,K", [(64, 2), (50, 2), (33, 2), (40, 1), (40, 0), (33, 0)])
def test_smooth_vorticity(native, g, K, kind):
    h = float(np.float32(1.0 / g))  # the cell size that the path computes with
    grid = (np.arange(g) + 0.5) / g
    pos = np.zeros((g ** 3, 4), np.float32)
    pos[:, 2], pos[:, 1], pos[:, 0] = (q.ravel() for q in np.meshgrid(grid, grid, grid, indexing="ij"))
    w = np.stack([f.ravel() * h ** 3 for f in _field(kind, g)])
    print(f"[far smooth] g={g} K={K} {kind}", flush=True)
    ctx = native.Context(native.config_params(g, K=K, precision=native.PREC_MIXED, mg_tol=1e-10))
    sc = native.Scene(pos, w)
    ctx.set_vortices(sc.n, sc.pos.ptr, sc.w_ptrs())
    ctx.compute_far_field()
    native.synchronize()
    psi, om, far = ([ctx.grid(which, c).reshape(g, g, g).astype(np.float64) for c in range(3)] for which in (1, 0, 2))
    assert max(np.abs(om[c] - w[c].reshape(g, g, g) / h ** 3).max() for c in range(3)) < 1e-5  # the field asked for

    def curl(f):
        d = lambda c, ax: np.subtract(*_clamped(f[c], ax)) * (0.5 / h)  # noqa: E731
        return [d(2, 1) - d(1, 0), d(0, 0) - d(2, 2), d(1, 2) - d(0, 1)]

    want = curl(psi)
    tol = [np.full((g, g, g), 2.0 ** -50 * max(np.abs(f).max() for f in psi) / h) for _ in range(3)]
    dc = DIAG * h * h
    for q, t in enumerate(curl([dc * f for f in om])):
        want[q] = want[q] - t
    for q, (a, b) in enumerate(((1, 2), (2, 0), (0, 1))):  # the components the curl's q takes differences of
        for f, ax in ((om[b], 2 - a), (om[a], 2 - b)):
            for nb in _clamped(f, ax):
                tol[q] = tol[q] + 4 * F32EPS * dc * 0.5 / h * np.abs(nb - f)
    inv = lambda *v: 1.0 / (FOUR_PI * h * np.sqrt(np.dot(v, v))) if any(v) else 0.0  # noqa: E731
    pad = [np.pad(f, max(K, 0)) for f in om]
    for k in range(-K, K + 1):
        for j in range(-K, K + 1):
            for i in range(-K, K + 1):
                if (i, j, k) == (0, 0, 0):
                    continue
                d = [0.5 / h * (inv(1 - i, -j, -k) - inv(-1 - i, -j, -k)) * h ** 3,
                     0.5 / h * (inv(-i, 1 - j, -k) - inv(-i, -1 - j, -k)) * h ** 3,
                     0.5 / h * (inv(-i, -j, 1 - k) - inv(-i, -j, -1 - k)) * h ** 3]
                o = [f[K + k:K + k + g, K + j:K + j + g, K + i:K + i + g] for f in pad]
                for q, (a, b) in enumerate(((1, 2), (2, 0), (0, 1))):
                    want[q] = want[q] - (d[a] * o[b] - d[b] * o[a])
                    tol[q] = tol[q] + 4 * F32EPS * (abs(d[a]) * np.abs(o[b] - om[b]) + abs(d[b]) * np.abs(o[a] - om[a]))
    for q in range(3):
        err, t = np.abs(far[q] - want[q]), tol[q] + 0.5 * np.spacing(np.abs(far[q]).astype(np.float32)) + 1e-30
        print(f"  component {q}: worst error / bound = {(err / t).max():.2f}", flush=True)
        assert (err <= t).all()
