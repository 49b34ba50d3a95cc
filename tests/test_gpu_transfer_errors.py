"""A HIP error that an earlier call left on the thread does not make a backend's
transfers fail: a spectra call too large for the device runs out of memory, then
a backend uploads and copies fields on the host's and the device's route."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(16, 16, 1), (128, 128, 8)])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_transfers_after_a_failed_allocation(fa, cells, precision):
    from fullmag_amd import _abi as A

    n = int(np.prod(cells))
    m = fa.generate_random_unit_vectors(3, n)
    b = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(3e-9, 3e-9, 3e-9), initial_magnetization=m[::-1].copy(),
                                       saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                       precision=precision, enable_demag=False))
    b.copy_field("H_ex")
    one = (ctypes.c_double * 1)()  # 691 GB of spectrum: fails before anything is written
    size = 60000
    rc = A.lib().fullmag_fdm_ext_newell_spectra(size, size, 1, 1e-9, 1e-9, 1e-9, 1, one, 6 * 2 * 4 * size * size)
    assert rc == A.FULLMAG_FDM_ERR_CUDA
    b.upload_magnetization(m)
    state = np.float32 if precision == "single" else np.float64
    np.testing.assert_array_equal(b.copy_field_f32("m"), m.astype(np.float32))
    np.testing.assert_array_equal(b.copy_field("m"), m.astype(state).astype(np.float64))
    b.close()
