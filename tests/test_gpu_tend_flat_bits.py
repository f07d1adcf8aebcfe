"""The Flat-z tendency kernel gives the bits of the thread-per-cell kernel in FP32 too, where the compiler fuses
what one expression holds: advection, constant diffusivity, rotation and tracers, each by itself and together."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import prognostic_names, uniform

pytestmark = pytest.mark.gpu

PHYSICS = {
    "plain": dict(),
    "viscous": dict(closure=om.ScalarDiffusivity(nu=0.3)),
    "rotating": dict(coriolis=om.FPlane(f=0.1)),
    "tracers": dict(closure=om.ScalarDiffusivity(nu=0.3, kappa=0.2), tracers=("c", "d"), coriolis=om.FPlane(f=0.1)),
}


@pytest.mark.parametrize("ft", [np.float32, np.float64])
@pytest.mark.parametrize("scheme", ["weno", "centered"])
@pytest.mark.parametrize("physics", PHYSICS)
@pytest.mark.parametrize("N", [(3, 4), (15, 15), (31, 45)], ids=lambda n: "x".join(map(str, n)))
def test_same_bits_as_the_cell_kernel(N, physics, scheme, ft):
    grid = om.RectilinearGrid(float_type=ft, size=N, x=(0, 3.0), y=(0, 2.0), topology=(om.Periodic, om.Periodic, om.Flat))
    kw = dict(PHYSICS[physics], advection=om.WENO() if scheme == "weno" else om.Centered())
    model = om.NonhydrostaticModel(grid, **kw)
    om.set_(model, **{n: uniform(7 + q, (*N, 1), -1, 1) for q, n in enumerate(prognostic_names(kw))})
    model.set_tuning(tendency_kernel="generic")
    model.update_state()
    ref = {n: f.interior().copy() for n, f in model.Gn.items()}
    model.set_tuning(tendency_kernel="tiled")
    model.update_state()
    for n, f in model.Gn.items():
        np.testing.assert_array_equal(f.interior(), ref[n], err_msg=f"G{n}")
    assert any(np.abs(v).max() > 0 for v in ref.values())
