"""The Fourier–tridiagonal solve of layers far wider than deep, whose columns are nearly singular (λ times the
depth down to 1e-10, far below 10·ε in FP32): every level is solved for, in both column kernels, at one and
two levels, in registers, in LDS, through memory and at the longest FP32 column.

The source is g(x, y) h(z) with h > 0, so that every sum of a column's elimination is over numbers of
one sign: at most 8·ε a level, beside 8·ε·log₂ n for each transform of the two there and back."""
import numpy as np
import pytest

import oceananigans_mi355x as om

pytestmark = pytest.mark.gpu

CASES = [(nz, ft) for nz in (1, 2, 12, 40, 67, 131, 316, 700) for ft in (np.float32, np.float64)] + [(16384, np.float32)]


@pytest.mark.parametrize("nz,ft", CASES, ids=lambda v: getattr(v, "__name__", str(v)))
def test_every_level_is_solved_for(nz, ft):
    nx, ny = (16, 8) if nz < 16384 else (4, 4)
    Lx, Ly = 2e6, 1.5e6
    rng = np.random.default_rng(nz)
    dz = 1 + rng.integers(0, 8, nz) / 16   # (faces, centres and spacings exact in FP32)
    faces = np.concatenate([[0.0], np.cumsum(dz)]) - dz.sum()
    grid = om.RectilinearGrid(float_type=ft, size=(nx, ny, nz), x=(0, Lx), y=(0, Ly), z=faces, topology=(om.Periodic, om.Periodic, om.Bounded))
    model = om.NonhydrostaticModel(grid, advection=om.Centered(), pressure_solver=om.FourierTridiagonalPoissonSolver())
    x, y = 2 * np.pi * np.arange(nx)[:, None] / nx, 2 * np.pi * np.arange(ny)[None, :] / ny
    g = np.cos(x + 0.3) + 0.7 * np.sin(y) + 0.5 * np.cos(x - y) + (0.2 * np.cos(2 * x + y + 1) if nx > 4 else 0)
    rhs = (g[:, :, None] * (1 + rng.random(nz))).astype(ft).astype(np.float64)
    p = model.poisson_solve(rhs)
    # the same columns from the bottom up in extended precision, the mean's column apart.  A pivot of the Thomas
    # algorithm is −(c[k + 1] + e) with e = Δz λ + c[k] e / (c[k] + e) of the level before: carried as e, since
    # the differences that otherwise form the pivots lose λ (1e-11 of them)
    ld = np.longdouble
    h = np.fft.fft2(rhs, axes=(0, 1)).astype(np.clongdouble)
    lam = lambda n, L: (2 * np.sin(np.pi * np.arange(n, dtype=ld) / n) * n / L) ** 2  # noqa: E731
    lxy, c = lam(nx, Lx)[:, None] + lam(ny, Ly)[None, :], np.zeros(nz + 1, ld)
    c[1:nz] = 2 / (dz[1:] + dz[:-1])
    lxy[0, 0] = 1   # (any: its source is zero)
    ratio, ref, e = np.zeros((nx, ny, nz), ld), np.zeros_like(h), 0
    for k in range(nz):
        e = dz[k] * lxy + (c[k] * e / (c[k] + e) if k else 0)
        pivot = c[k + 1] + e
        ratio[..., k] = c[k + 1] / pivot
        ref[..., k] = ((c[k] * ref[..., k - 1] if k else 0) - dz[k] * h[..., k]) / pivot
    for k in range(nz - 2, -1, -1):
        ref[..., k] += ratio[..., k] * ref[..., k + 1]
    ref[0, 0] = 0
    ref = np.fft.ifft2(ref.astype(np.complex128), axes=(0, 1)).real
    err = np.abs(p - ref).max() / np.abs(ref).max()
    tol = np.finfo(ft).eps * (16 * (np.log2(nx) + np.log2(ny)) + 8 * nz)
    print(nz, np.dtype(ft).name, f"{err:.2e} <= {tol:.2e}", flush=True)
    assert err <= tol
