"""The Fourier–tridiagonal solve at the sizes where its two-ended column elimination can go wrong: one,
two and three levels, an odd and even number, whole batches and remainders of either precision, and
columns so long that they pass through memory.

Each column is eliminated backward-stably and the transforms are unitary up to 8·ε·log₂ n each way, so
the solution's residual stays within that share of ‖L‖₂‖p‖₂ (16·ε more for the columns and the rounding
of p itself)."""
import numpy as np
import pytest

import oceananigans_mi355x as om

pytestmark = pytest.mark.gpu

SIZES = [(8, 6, 1), (8, 6, 2), (6, 8, 3), (16, 16, 15), (16, 16, 16), (40, 6, 17), (32, 8, 31), (33, 9, 32), (32, 10, 33), (48, 20, 34), (8, 8, 64),
         (34, 12, 65), (70, 66, 67), (16, 8, 341), (16, 4, 342), (8, 4, 700), (4, 4, 3000), (4, 3, 8192)]


@pytest.mark.parametrize("ft", [np.float32, np.float64])
@pytest.mark.parametrize("N", SIZES, ids=lambda n: "x".join(map(str, n)))
def test_residual(N, ft):
    nx, ny, nz = N
    rng = np.random.default_rng(sum(N))
    faces = np.concatenate([[0.0], np.cumsum(1 + 0.3 * rng.random(nz))])
    faces -= faces[-1]
    grid = om.RectilinearGrid(float_type=ft, size=N, x=(0, nx), y=(0, ny), z=faces, topology=(om.Periodic, om.Periodic, om.Bounded))
    advection = om.WENO() if min(N) >= 3 else om.Centered()
    model = om.NonhydrostaticModel(grid, advection=advection, pressure_solver=om.FourierTridiagonalPoissonSolver())
    dzc = np.diff(faces)
    rhs = rng.standard_normal(N)
    rhs -= (rhs * dzc).sum() / (nx * ny * dzc.sum())   # solvable: no volume integral
    rhs = rhs.astype(ft).astype(np.float64)
    p = model.poisson_solve(rhs)
    zc = 0.5 * (faces[1:] + faces[:-1])
    flux = np.zeros((nx, ny, nz + 1))
    flux[:, :, 1:-1] = np.diff(p, axis=2) / np.diff(zc)
    L = sum(np.roll(p, 1, a) - 2 * p + np.roll(p, -1, a) for a in (0, 1)) + np.diff(flux, axis=2) / dzc
    norm = 8 + (4 / (dzc.min() ** 2) if nz > 1 else 0)
    eps = np.finfo(ft).eps
    tol = eps * (8 * 2 * (np.log2(nx) + np.log2(ny)) + 16)
    err = np.linalg.norm(L - rhs) / (norm * np.linalg.norm(p))
    print(N, np.dtype(ft).name, f"{err:.2e} <= {tol:.2e}", flush=True)
    assert np.isfinite(p).all()
    assert err <= tol
    assert abs(p.mean()) <= 16 * eps * np.abs(p).max()
