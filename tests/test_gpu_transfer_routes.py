"""Whole-field transfers on both sides of the cell counts from which the device
converts them: the state round-trips bit for bit in every pairing of precisions,
with inactive cells zero, and small fields leave no scratch behind."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the edges of the rules, one cell below and at: uploads 16384, 32768, 98304;
# copies 24576, 45056, 81920, 2621440
COUNTS = [16383, 16384, 24575, 24576, 32767, 32768, 45055, 45056, 81919, 81920, 98303, 98304, 2621439, 2621440]


def backend(fa, n, precision, mask):
    return fa.NativeFdmBackend(fa.FdmPlan(cells=(n, 1, 1), cell_size=(3e-9, 3e-9, 3e-9),
                                          initial_magnetization=np.tile([0.0, 0.0, 1.0], (n, 1)),
                                          saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                          precision=precision, enable_demag=False, active_mask=mask))


@pytest.mark.parametrize("n", COUNTS)
@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
def test_round_trip_at_the_edges(fa, n, precision):
    rng = np.random.default_rng(n)
    mask = (rng.random(n) < 0.7).astype(np.uint8)
    b = backend(fa, n, precision, mask)
    m = rng.standard_normal((n, 3))
    state = np.float32 if precision == "single" else np.float64
    for up, src in ((b.upload_magnetization, m), (b.upload_magnetization_f32, m.astype(np.float32))):
        up(src)
        want = np.where(mask[:, None] != 0, src.astype(state), state(0))
        np.testing.assert_array_equal(b.copy_field("m"), want.astype(np.float64))
        np.testing.assert_array_equal(b.copy_field_f32("m"), want.astype(np.float32))
    if precision == "mixed":  # an FP32 field of an FP64 state
        np.testing.assert_array_equal(b.copy_field("H_ex").astype(np.float32), b.copy_field_f32("H_ex"))
    b.close()


@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
def test_small_transfers_need_no_scratch(fa, precision):
    """The arrays of two small backends differ by their cells' share and the
    reductions' partials (72 bytes per 64 cells), not by the 24 bytes per cell of
    a scratch, and transfers add nothing."""
    a, b = backend(fa, 64, precision, None), backend(fa, 8192, precision, None)
    state, real = (4 if precision == "single" else 8), (8 if precision == "double" else 4)
    per_cell = 3 * (state + 4 * real)  # m, one slope, one stage point, H_ex and H_eff
    for x in (a, b):
        x.copy_field("H_ex")  # an upload keeps the fields of the state before it
    held = [x.device_bytes() for x in (a, b)]
    assert 0 <= held[1] - held[0] - (8192 - 64) * per_cell <= 2 * (8192 - 64)
    for x, h in zip((a, b), held):
        x.upload_magnetization(x.copy_field("m"))
        x.upload_magnetization_f32(x.copy_field_f32("m"))
        assert x.device_bytes() == h
        x.close()
