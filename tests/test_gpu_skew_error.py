"""FP32 rounding of the demag field at the x frequencies k + 1/2 against the
integer ones, for a smooth state, whose mean the shifted frequencies spread over
the whole spectrum.

Bound: both plans round their inputs once.  The shifted one multiplies its
outputs by FP32 factors as well, two roundings of 2^-24 of a field whose error
is about five of them (2 % in quadrature), and its table roots meet the spread
mean (5 to 8 % in a plain FP32 transform of the same sizes).  15 % of the rms
error is allowed.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def smooth_state(nx, ny, nz):
    y, x = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    th = 0.4 * np.sin(2 * np.pi * x / nx + 0.7) + 0.2 * np.cos(2 * np.pi * y / ny)
    v = np.stack([np.cos(th), np.sin(th), np.full(th.shape, 0.1)], -1)
    v /= np.linalg.norm(v, axis=-1, keepdims=True)
    return np.broadcast_to(v[None], (nz, ny, nx, 3)).reshape(-1, 3)


@pytest.mark.parametrize("precision", ["mixed", "single"])
@pytest.mark.parametrize("cells", [(128, 128, 4), (128, 128, 8), (256, 256, 4), (200, 30, 2)])
def test_shifted_frequencies_round_as_integer_ones(fa, monkeypatch, cells, precision):
    m = smooth_state(*cells)

    def field(prec, tune):
        monkeypatch.setenv("FULLMAG_FDM_TUNE", tune)
        gpu = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(4e-9, 4e-9, 2e-9), initial_magnetization=m,
                                             saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                             precision=prec, demag_kernel="device"))
        h = gpu.copy_h_demag()
        gpu.close()
        return h

    ref = field("double", "")
    rms = [float(np.sqrt(((field(precision, tune) - ref) ** 2).mean())) for tune in ("", "skew=0")]
    assert rms[0] <= 1.15 * rms[1]
