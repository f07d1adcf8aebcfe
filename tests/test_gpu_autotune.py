"""The autotuner keeps the chunk that a kernel has where none of its candidates is faster: the closure kernel
after tuning against before, on grids whose chunk by size is not among the round numbers (at 32³ it is one level)."""
import numpy as np
import pytest

from cases import convection, product_for

pytestmark = pytest.mark.gpu


def closure_us(model):
    model.set_phase_timing(True)
    best = np.inf
    for _ in range(7):
        model.time_step(0.5, 4)
        ms, n = model.phase_times()["closure"]
        best = min(best, 1e3 * ms / n)
    model.set_phase_timing(False)
    return best


@pytest.mark.parametrize("N", [(32, 32, 32), (64, 64, 64), (150, 100, 75)], ids=lambda n: "x".join(map(str, n)))
def test_tuned_closure_is_no_slower(N):
    model = product_for(*convection(N=N, float_type=np.float32, noise_velocity=1e-2))
    model.time_step(0.5, 2)
    before = closure_us(model)
    nu = model.closure_fields["nu"].interior().copy()
    model.autotune()
    np.testing.assert_array_equal(model.closure_fields["nu"].interior(), nu)
    after = closure_us(model)
    print(N, f"{before:.1f} -> {after:.1f} us", flush=True)
    assert after <= 1.15 * before
