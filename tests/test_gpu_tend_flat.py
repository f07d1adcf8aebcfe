"""The Flat-z tendency kernel, which evaluates each face flux once, against the thread-per-cell kernel: equal
in FP64, within FP32 rounding in FP32 (there the difference of two area-weighted viscous fluxes fuses
differently: a few ε of the largest tendency, held to 1e-5 like the other tiled kernels), on grids
smaller than a tile, of whole tiles and with remainders; with w carried by the flow, constant
diffusivity, tracers, rotation; and against the oracle."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import oracle_for, prognostic_names, rel_err, uniform

pytestmark = pytest.mark.gpu

PHYSICS = {
    "plain": dict(),
    "viscous": dict(closure=om.ScalarDiffusivity(nu=0.3)),
    "tracers": dict(closure=om.ScalarDiffusivity(nu=0.3, kappa=0.2), tracers=("c", "d"), coriolis=om.FPlane(f=0.1)),
}


def build(N, physics, advection, ft):
    grid = om.RectilinearGrid(float_type=ft, size=N, x=(0, 3.0), y=(0, 2.0), topology=(om.Periodic, om.Periodic, om.Flat))
    kw = dict(PHYSICS[physics], advection=advection)
    init = {n: uniform(7 + q, (*N, 1), -1, 1) for q, n in enumerate(prognostic_names(kw))}
    return grid, kw, init


@pytest.mark.parametrize("ft", [np.float32, np.float64])
@pytest.mark.parametrize("scheme", ["weno", "centered"])
@pytest.mark.parametrize("physics", PHYSICS)
@pytest.mark.parametrize("N", [(3, 4), (15, 15), (16, 14), (31, 45), (64, 17)], ids=lambda n: "x".join(map(str, n)))
def test_equals_the_cell_kernel(N, physics, scheme, ft):
    grid, kw, init = build(N, physics, om.WENO() if scheme == "weno" else om.Centered(), ft)
    model = om.NonhydrostaticModel(grid, **kw)
    om.set_(model, **init)
    model.set_tuning(tendency_kernel="generic")
    model.update_state()
    ref = {n: f.interior().copy() for n, f in model.Gn.items()}
    model.set_tuning(tendency_kernel="tiled")
    model.update_state()
    for n, f in model.Gn.items():
        if ft is np.float64:
            np.testing.assert_array_equal(f.interior(), ref[n], err_msg=f"G{n}")
        else:
            assert rel_err(f.interior(), ref[n]) <= 1e-5, n
    assert any(np.abs(v).max() > 0 for v in ref.values())


@pytest.mark.parametrize("physics", ["plain", "tracers"])
def test_steps_match_the_oracle(physics):
    grid, kw, init = build((20, 18), physics, om.WENO(), np.float64)
    init.pop("w")
    model = om.NonhydrostaticModel(grid, **kw)
    om.set_(model, **init)
    orc = oracle_for(grid, kw, init)
    model.time_step(1e-3, 2)
    orc.time_step(1e-3, 2)
    for q, n in enumerate(prognostic_names(kw)):
        f = model.velocities[n] if n in "uvw" else model.tracers[n]
        assert rel_err(f.interior(), orc.get(q)) <= 1e-12, n
