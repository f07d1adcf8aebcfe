"""The hydrostatic pressure anomaly's column scans at the edges of their slabs (FP64: 64 levels, eight
per wave) and segments (FP32: eight or sixteen of up to 16 levels), on rows longer than a block, for a
buoyancy tracer and for temperature and salinity, uniform and stretched z.

FP64 sums in the oracle's order: equal to rounding of the same operations, bit for bit.  FP32 sums in
segments: relative to the largest anomaly within 32 rounding errors of a sum of this many terms' size."""
import numpy as np
import pytest

import oceananigans_mi355x as om
from cases import convection, oracle_for, product_for, stretched_convection, wind_convection

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [convection, wind_convection, stretched_convection])
@pytest.mark.parametrize("nz", [3, 8, 9, 63, 64, 65, 72, 128, 129, 200])
def test_fp64_scan_equals_the_oracle(nz, make):
    grid, kw, init = make(N=(70, 5, nz), float_type=np.float64)
    model = product_for(grid, kw, init)
    orc = oracle_for(grid, kw, init)
    np.testing.assert_array_equal(model.pressures.pHY.interior(), orc.get(om._abi.OM_FIELD_PHY))


@pytest.mark.parametrize("make", [convection, wind_convection, stretched_convection])
@pytest.mark.parametrize("nz", [3, 8, 9, 15, 16, 17, 113, 128, 129, 200, 256])
def test_fp32_scan_matches_the_oracle(nz, make):
    grid, kw, init = make(N=(70, 5, nz), float_type=np.float32)
    model = product_for(grid, kw, init)
    orc = oracle_for(grid, kw, init, oracle_float_type=np.float64, round_inputs_to=np.float32)
    a, b = model.pressures.pHY.interior(), orc.get(om._abi.OM_FIELD_PHY)
    assert np.abs(a - b).max() <= 32 * np.finfo(np.float32).eps * np.abs(b).max()
