"""Steps taken one call at a time, which replay a captured step once Δt has stayed the same for a while,
against the same steps launched directly: every bit, over both buffer assignments, through changes of Δt,
calls of several steps, a tuning change and a state set anew in between."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import convection, prognostic_names, product_for

pytestmark = pytest.mark.gpu

CALLS = [(1.0, 1)] * 12 + [(0.5, 1)] * 3 + [(1.0, 1)] * 9 + [(1.0, 3)] * 3 + [(1.0, 2)] * 2 + [(1.0, 1)] * 5 + [(0.25, 1)] * 11


@pytest.mark.parametrize("ft", [np.float32, np.float64])
def test_replayed_single_steps_equal_direct_ones(ft):
    grid, kw, init = convection(N=(16, 12, 8), float_type=ft)
    graph, direct = product_for(grid, kw, init), product_for(grid, kw, init)
    direct.set_tuning(step_graphs=False)
    names = prognostic_names(kw)

    def fields(m):
        return {**{n: (m.velocities[n] if n in "uvw" else m.tracers[n]).interior().copy() for n in names}, "p": m.pressures.pNHS.interior().copy()}

    for q, (dt, n) in enumerate(CALLS):
        if q == 20:
            for m in (graph, direct):
                m.set_tuning(kchunk=3)
        if q == 33:
            for m in (graph, direct):
                om.set_(m, b=lambda x, y, z: 1e-5 * z)
        for m in (graph, direct):
            m.time_step(dt, n)
        a, b = fields(graph), fields(direct)
        for c in a:
            np.testing.assert_array_equal(a[c], b[c], err_msg=f"call {q}: {c}")
    assert np.isfinite(a["u"]).all() and np.abs(a["w"]).max() > 0
