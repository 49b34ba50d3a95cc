"""Whole-field transfers: the state round-trips bit for bit through upload and
copy in every pairing of precisions, with inactive cells zero, below and above
the cell count converted per pass (2^21)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1, 1, 1), (7, 5, 3), (257, 1, 1), (1500, 1400, 1)])
@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
@pytest.mark.parametrize("masked", [False, True])
def test_state_round_trip(fa, cells, precision, masked):
    n = int(np.prod(cells))
    rng = np.random.default_rng(n)
    mask = (rng.random(n) < 0.7).astype(np.uint8) if masked else None
    b = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(3e-9, 3e-9, 3e-9),
                                       initial_magnetization=np.tile([0.0, 0.0, 1.0], (n, 1)),
                                       saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                       precision=precision, enable_demag=False, active_mask=mask))
    m = rng.standard_normal((n, 3))
    state = np.float32 if precision == "single" else np.float64
    keep = np.ones((n, 1)) if mask is None else mask.reshape(n, 1).astype(np.float64)
    for up, src in ((b.upload_magnetization, m), (b.upload_magnetization_f32, m.astype(np.float32))):
        up(src)
        want = (src.astype(state) * keep).astype(state)
        np.testing.assert_array_equal(b.copy_field("m"), want.astype(np.float64))
        np.testing.assert_array_equal(b.copy_field_f32("m"), want.astype(np.float32))
    b.close()
