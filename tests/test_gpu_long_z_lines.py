"""The longest z lines of the FFT pressure solver: an odd Bounded Nz is one transform of that length, as an even
one is, so it is accepted up to the same limit (2047 levels in FP32, 1023 in FP64), and refused beyond."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from test_gpu_fft_lengths import reference

pytestmark = pytest.mark.gpu


def build(nz, ft, ztop=om.Bounded):
    grid = om.RectilinearGrid(float_type=ft, size=(6, 4, nz), x=(0, 6), y=(0, 4), z=(-nz, 0), topology=(om.Periodic, om.Periodic, ztop))
    return om.NonhydrostaticModel(grid, advection=om.WENO())


@pytest.mark.parametrize("nz,ft", [(1365, np.float32), (1367, np.float32), (1501, np.float32), (2046, np.float32), (2047, np.float32),
                                   (683, np.float64), (1001, np.float64), (1023, np.float64)])
def test_odd_lengths_solve(nz, ft):
    rhs = np.random.default_rng(nz).standard_normal((6, 4, nz))
    rhs = (rhs - rhs.mean()).astype(ft).astype(np.float64)
    got, ref = build(nz, ft).poisson_solve(rhs), reference(rhs, om.Bounded)
    err = np.abs(got - ref).max() / np.abs(ref).max()
    tol = 8 * np.finfo(ft).eps * sum(np.log2(n) for n in (6, 4, nz))
    print(nz, np.dtype(ft).name, f"{err:.2e} <= {tol:.2e}", flush=True)
    assert err <= tol


@pytest.mark.parametrize("nz,ft", [(2049, np.float32), (2050, np.float32), (1025, np.float64), (1026, np.float64)])
def test_longer_ones_are_refused(nz, ft):
    with pytest.raises(om.OmError, match="64 KiB"):
        build(nz, ft)
