"""The FP32 pressure correction of a nearly divergence-free flow, whose velocity differences cancel to a
thousandth of each, against the FP64 one of the same FP32 velocities.

On grids with a line that is not a power of two the divergence is rounded nearly once, so the pressure is as
accurate as its transforms: 8·ε·Σ log₂ n.  Where all lines are powers of two each of the six products
and the sums round on their own: white noise of up to 8·ε·max|U| a cell, which the inverse Laplacian
amplifies by at most 1/λ of the longest wave."""
import numpy as np
import pytest

import oceananigans_mi355x as om

pytestmark = pytest.mark.gpu


def flow(N, ztop):
    """u, v, w on their faces (unit spacing): the discrete curl of a random potential plus a thousandth of noise."""
    rng = np.random.default_rng(sum(N))
    bounded, flat = ztop is om.Bounded, ztop is om.Flat
    ax, ay, az = (rng.standard_normal(N) for _ in range(3))
    if bounded:
        ax[:, :, 0] = ay[:, :, 0] = 0
    d = lambda a, q: np.roll(a, -1, q) - a  # noqa: E731
    if flat:
        ax, ay = 0 * ax, 0 * ay

    def dz(a):   # above the top the potential vanishes (Bounded) or wraps
        return np.concatenate([a[:, :, 1:], 0 * a[:, :, :1]], 2) - a if bounded else d(a, 2)

    U = [d(az, 1) - dz(ay), dz(ax) - d(az, 0), d(ay, 0) - d(ax, 1)]
    U = [u + 1e-3 * rng.standard_normal(N) for u in U]
    if bounded:
        U[2][:, :, 0] = 0
    if flat:
        U[2] = 0 * U[2]
    return [u.astype(np.float32).astype(np.float64) for u in U]


@pytest.mark.parametrize("ztop", [om.Bounded, om.Periodic, om.Flat], ids=["bounded", "periodic", "flat"])
@pytest.mark.parametrize("N", [(24, 20, 10), (15, 16, 8), (16, 9, 8), (16, 16, 7), (32, 16, 8)], ids=lambda n: "x".join(map(str, n)))
def test_pressure_of_a_nearly_divergence_free_flow(N, ztop):
    flat = ztop is om.Flat
    n = (*N[:2], 1) if flat else N
    U = flow(n, ztop)
    p = {}
    for ft in (np.float32, np.float64):
        grid = om.RectilinearGrid(float_type=ft, size=n[:2] if flat else n, x=(0, n[0]), y=(0, n[1]), topology=(om.Periodic, om.Periodic, ztop),
                                  **({} if flat else dict(z=(-n[2], 0))))
        model = om.NonhydrostaticModel(grid, advection=om.WENO())
        for c, u in zip("uvw", U):
            model.set_interior(c, u)
        model.compute_pressure_correction(1.0)
        p[ft] = model.pressures.pNHS.interior().copy()
    ref, eps = p[np.float64], np.finfo(np.float32).eps
    err = np.linalg.norm(p[np.float32] - ref) / np.linalg.norm(ref)
    tol = 8 * eps * sum(np.log2(max(m, 2)) for m in n)
    if all(m & (m - 1) == 0 for m in n):
        noise = 8 * eps * max(np.abs(u).max() for u in U) * np.sqrt(np.prod(n))
        tol += noise * (max(n[0], n[1], 2 * n[2]) / 4) ** 2 / np.linalg.norm(ref)   # (sin x ≥ 2x/π: λ ≥ (4/n)²)
    print(n, ztop.__name__, f"{err:.2e} <= {tol:.2e}", flush=True)
    assert err <= tol
