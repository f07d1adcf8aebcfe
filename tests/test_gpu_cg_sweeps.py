"""The sweeps of the conjugate-gradient solver at the edges of their tiles (64 × 8 columns) and chunks: one
row, column and level more or less than a tile, the smallest grids, several tiles and chunks with remainders;
with and without an immersed bottom.  Bars as in test_gpu_cg.py: FP64 solutions within 1e-11 of the
oracle's at reltol = 1e-13."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import oracle_for, rel_err, seamount

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("immersed", [True, False])
@pytest.mark.parametrize("N", [(4, 3, 4), (63, 7, 7), (64, 8, 8), (65, 9, 9), (16, 17, 33), (130, 16, 12)], ids=lambda n: "x".join(map(str, n)))
def test_solve_matches_oracle(N, immersed):
    from oceananigans_mi355x.synthetic import uniform
    grid, kw, _ = seamount(N=N)
    if not immersed:
        grid = om.RectilinearGrid(float_type=np.float64, size=N, x=(0, 10e3), y=(0, 10e3), z=grid.z_faces)
    pc = om.FourierTridiagonalPoissonSolver()
    kw = dict(kw, pressure_solver=om.ConjugateGradientPoissonSolver(preconditioner=pc, reltol=1e-13, abstol=0))
    model = om.NonhydrostaticModel(grid, **kw)
    orc = oracle_for(grid, kw, {})
    dz = np.diff(grid.z_faces)
    V = np.broadcast_to(dz[None, None, :], N)
    rhs = uniform(21, N, -1, 1)
    wet = np.ones(N, bool)
    if immersed:
        H = grid.H[2]
        wet = orc.grid_z()[2][H:H + N[2]][None, None, :] > grid.bottom_heights()[:, :, None]
        rhs[~wet] = 0
    rhs[wet] -= (V * rhs)[wet].sum() / V[wet].sum()
    phi, phi_o = model.poisson_solve(rhs), orc.poisson_solve(rhs)
    e = rel_err(phi, phi_o)
    print(N, immersed, "iterations", model.last_solve_info()[0], orc.last_solve_info()[0], f"rel err {e:.1e}", flush=True)
    assert e <= 1e-11
