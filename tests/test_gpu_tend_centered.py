"""The z-marching kernel of Centered(order=2) advection against the thread-per-cell kernel: identically
rounded tendencies for every combination it covers (Bounded and Periodic z, constant diffusivity or
none, no, one or two tracers, buoyancy with and without a hydrostatic pressure, rotation, halos of one
cell and more), on grids smaller than a tile, with tile and chunk remainders; and against the oracle."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import oracle_for, prognostic_names, rel_err, uniform

pytestmark = pytest.mark.gpu

PHYSICS = {
    "plain": dict(),
    "viscous": dict(closure=om.ScalarDiffusivity(nu=0.3)),
    "tracer": dict(closure=om.ScalarDiffusivity(nu=0.3, kappa=0.2), tracers=("c",)),
    "buoyant": dict(closure=om.ScalarDiffusivity(nu=0.3, kappa=0.2), tracers=("c", "b"), buoyancy=om.BuoyancyTracer(), coriolis=om.FPlane(f=0.1)),
    "seawater": dict(tracers=("T", "S"), buoyancy=om.SeawaterBuoyancy(equation_of_state=om.LinearEquationOfState(2e-4, 8e-4)),
                     coriolis=om.FPlane(f=0.1), hydrostatic_pressure_anomaly=None),
}


def build(N, ztop, physics, ft, halo):
    grid = om.RectilinearGrid(float_type=ft, size=N, x=(0, 3.0), y=(0, 2.0), z=(-1.5, 0), topology=(om.Periodic, om.Periodic, ztop), halo=(halo,) * 3)
    kw = dict(PHYSICS[physics])
    if ztop is om.Periodic and physics == "buoyant":
        kw["hydrostatic_pressure_anomaly"] = None
    init = {n: uniform(7 + q, N, -1, 1) for q, n in enumerate(prognostic_names(kw)) if n != "w" or ztop is om.Periodic}
    return grid, kw, init


@pytest.mark.parametrize("ft", [np.float32, np.float64])
@pytest.mark.parametrize("physics", PHYSICS)
@pytest.mark.parametrize("ztop", [om.Bounded, om.Periodic], ids=["bounded", "periodic"])
@pytest.mark.parametrize("N,halo", [((3, 2, 4), 2), ((32, 8, 5), 3), ((33, 9, 17), 2), ((47, 30, 12), 3)], ids=lambda n: str(n))
def test_march_rounds_like_the_cell_kernel(N, halo, ztop, physics, ft):
    grid, kw, init = build(N, ztop, physics, ft, halo)
    model = om.NonhydrostaticModel(grid, **kw)
    om.set_(model, **init)
    model.set_tuning(tendency_kernel="generic")
    model.update_state()
    ref = {n: f.interior().copy() for n, f in model.Gn.items()}
    model.set_tuning(tendency_kernel="tiled")
    for kchunk in (1, 3, N[2]):
        model.set_tuning(kchunk=kchunk)
        model.update_state()
        for n, f in model.Gn.items():
            np.testing.assert_array_equal(f.interior(), ref[n], err_msg=f"G{n}, chunk {kchunk}")
    assert any(np.abs(v).max() > 0 for v in ref.values())


@pytest.mark.parametrize("ztop", [om.Bounded, om.Periodic], ids=["bounded", "periodic"])
def test_step_matches_the_oracle(ztop):
    grid, kw, init = build((20, 12, 10), ztop, "buoyant", np.float64, 3)
    model = om.NonhydrostaticModel(grid, **kw)
    om.set_(model, **init)
    orc = oracle_for(grid, kw, init)
    model.time_step(1e-3, 2)
    orc.time_step(1e-3, 2)
    for q, n in enumerate(prognostic_names(kw)):
        f = model.velocities[n] if n in "uvw" else model.tracers[n]
        assert rel_err(f.interior(), orc.get(q)) <= 1e-12, n
