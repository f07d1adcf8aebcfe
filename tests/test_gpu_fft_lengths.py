"""Pressure solves on grids whose lines are not powers of two: every radix of the mixed-radix
transform (2, 3, 4, 5, 7 and primes above 7 as direct sums), odd and even x and z, prime lines, the
smallest lines and the longest that both precisions accept, on Bounded, Periodic and Flat z.

The reference is the same discrete problem solved in FP64 by scipy's FFT and DCT.  Tolerances, set
beforehand: an FFT's error grows as ε·log₂ n per transform, two transforms per axis, each a few ε
worst case: 8·ε·Σ log₂ n relative to the largest value."""
import numpy as np
import pytest
import scipy.fft

import oceananigans_mi355x as om

pytestmark = pytest.mark.gpu

SIZES = [(6, 3, 5), (3, 5, 3), (10, 14, 7), (9, 6, 12), (18, 22, 9), (26, 30, 15), (34, 21, 25), (96, 60, 27), (150, 49, 75),
         (13, 11, 3), (210, 33, 35), (254, 17, 127), (64, 48, 45), (49, 64, 121), (2730, 3, 4)]


def reference(rhs, ztop):
    nx, ny, nz = rhs.shape
    # sin(πm/n) from the nearer end: near m = n, π's own rounding would be a relative error of n·ε
    lam = lambda n: (2 * np.sin(np.pi * np.minimum(np.arange(n), n - np.arange(n)) / n)) ** 2
    h = scipy.fft.fftn(rhs, axes=(0, 1))
    den = lam(nx)[:, None, None] + lam(ny)[None, :, None] + 0 * h.real
    if ztop is om.Periodic:
        h = scipy.fft.fft(h, axis=2)
        den = den + lam(nz)[None, None, :]
    elif ztop is om.Bounded:
        h = scipy.fft.dct(h.real, axis=2) + 1j * scipy.fft.dct(h.imag, axis=2)
        den = den + ((2 * np.sin(np.pi * np.arange(nz) / (2 * nz))) ** 2)[None, None, :]
    den[0, 0, 0] = 1
    h = -h / den
    h[0, 0, 0] = 0
    if ztop is om.Periodic:
        h = scipy.fft.ifft(h, axis=2)
    elif ztop is om.Bounded:
        h = scipy.fft.idct(h.real, axis=2) + 1j * scipy.fft.idct(h.imag, axis=2)
    return scipy.fft.ifftn(h, axes=(0, 1)).real


@pytest.mark.parametrize("ft", [np.float32, np.float64])
@pytest.mark.parametrize("ztop", [om.Bounded, om.Periodic, om.Flat], ids=["bounded", "periodic", "flat"])
@pytest.mark.parametrize("N", SIZES, ids=lambda n: "x".join(map(str, n)))
def test_solve_matches_fp64_transforms(N, ztop, ft):
    flat = ztop is om.Flat
    n = (N[0], N[1], 1) if flat else N
    grid = om.RectilinearGrid(float_type=ft, size=n[:2] if flat else n, x=(0, n[0]), y=(0, n[1]), topology=(om.Periodic, om.Periodic, ztop),
                              **({} if flat else dict(z=(-n[2], 0))))
    model = om.NonhydrostaticModel(grid, advection=om.WENO())
    rhs = np.random.default_rng(sum(n)).standard_normal(n).astype(ft).astype(np.float64)
    rhs -= rhs.mean()
    rhs = rhs.astype(ft).astype(np.float64)
    ref = reference(rhs, ztop)
    got = model.poisson_solve(rhs)
    err = np.abs(got - ref).max() / np.abs(ref).max()
    tol = 8 * np.finfo(ft).eps * sum(np.log2(max(v, 2)) for v in n)
    print(N, ztop.__name__, np.dtype(ft).name, f"{err:.2e} <= {tol:.2e}", flush=True)
    assert err <= tol
