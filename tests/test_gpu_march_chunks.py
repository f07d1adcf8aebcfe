"""The tiled kernels' z chunk is chosen by the grid's size; the choice changes no result: tendencies,
viscosity and diffusivity of the default equal those of explicit chunks bit for bit, on grids smaller
than a tile, with ragged tile and chunk remainders, and with chunks longer than the column."""
import numpy as np
import pytest

from cases import convection, product_for, wind_convection

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ft", [np.float32, np.float64])
@pytest.mark.parametrize("make", [convection, wind_convection])
@pytest.mark.parametrize("N", [(5, 4, 3), (16, 15, 7), (31, 33, 40), (64, 64, 64), (46, 75, 65)], ids=lambda n: "x".join(map(str, n)))
def test_default_chunk_changes_no_result(N, make, ft):
    grid, kw, init = make(N=N, float_type=ft)
    model = product_for(grid, kw, init)
    fields = {**{"G" + n: f for n, f in model.Gn.items()}, "nu": model.closure_fields["nu"]}
    ref = {n: f.interior().copy() for n, f in fields.items()}
    chosen = model.get_tuning()["kchunk"]
    assert 1 <= chosen <= N[2]
    for kchunk in (1, 3, N[2] + 2):
        model.set_tuning(kchunk=kchunk)
        model.update_state()
        for n, f in fields.items():
            assert np.isfinite(ref[n]).all()
            np.testing.assert_array_equal(f.interior(), ref[n], err_msg=f"{n} at chunk {kchunk} against {chosen}")
