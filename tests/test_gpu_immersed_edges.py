"""The immersed bottom's tables at their edges: rough bottoms (every buffer rule next to every other),
columns without and full of immersed cells, grids narrower than a stencil and than a tile of the
fix-up launches.  Bars as in test_gpu_immersed.py: FP64 tendencies and closure fields on identical inputs
within 1e-12 of the oracle's."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import prognostic_names, rel_err, seamount
from test_gpu_parity import compare_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["tiled", "generic"])
@pytest.mark.parametrize("N", [(3, 4, 8), (5, 3, 9), (16, 4, 12), (17, 9, 10), (33, 15, 24)], ids=lambda n: "x".join(map(str, n)))
def test_rough_bottom_tendencies_fp64(N, kernel):
    from oracle.oracle import OracleModel
    _, kw, init = seamount(N=N)
    rng = np.random.default_rng(sum(N))
    bottom = np.where(rng.random(N[:2]) < 0.6, -1000.0 + 700.0 * rng.random(N[:2]) ** 2, -1100.0)
    bottom[0, 0] = -50.0
    under = om.RectilinearGrid(float_type=np.float64, size=N, x=(0, 10e3), y=(0, 10e3), z=(-1000.0, 0))
    grid = om.ImmersedBoundaryGrid(under, om.GridFittedBottom(bottom))
    model = om.NonhydrostaticModel(grid, **kw)
    model.set_tuning(tendency_kernel=kernel)
    om.set_(model, enforce_incompressibility=False, **init)
    cfg, keep = om.build_config(grid, **kw)
    orc = OracleModel(cfg, grid)
    names = prognostic_names(kw)
    for name, val in init.items():
        orc.set(names.index(name), om.models._evaluate(grid, name, val))
    orc.set_finalize(False)
    compare_state(model, orc, kw, fields=("state", "G"), label=f"rough {N}")
    assert rel_err(model.closure_fields.nu.interior(), orc.get(om._abi.OM_FIELD_NU)) <= 1e-12
    assert rel_err(model.closure_fields.kappa_b.interior(), orc.get(om._abi.OM_FIELD_KAPPA0)) <= 1e-12
