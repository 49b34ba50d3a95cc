"""Transform lengths above 1024 points: cells that pad to 2048 and 4096, where
the general path at 2n gives the reference field (FP64, runtime plans), at both
ends of the range of each length, along each axis, films, slabs and long z lines.
Bars of test_gpu_lengths.py: 1e-12 of the largest value in FP64, 2e-6 in FP32."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BAR = {"double": 1e-12, "mixed": 2e-6}


def demag_field(fa, monkeypatch, cells, precision, tune):
    monkeypatch.setenv("FULLMAG_FDM_TUNE", tune)
    n = int(np.prod(cells))
    gpu = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(4e-9, 3e-9, 2e-9),
                                         initial_magnetization=fa.generate_random_unit_vectors(71 + n, n),
                                         saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                         precision=precision, demag_kernel="device"))
    h = gpu.copy_h_demag()
    gpu.close()
    return h


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("cells", [(768, 5, 1), (5, 768, 1), (1000, 12, 3), (7, 1023, 2), (1023, 6, 1), (9, 1000, 1),
                                   (1024, 4, 2), (4, 1024, 5), (1536, 5, 1), (6, 1536, 2), (2000, 3, 2), (3, 2047, 1),
                                   (2048, 4, 1), (4, 2048, 2), (4, 3, 768), (3, 4, 1000), (600, 9, 1), (9, 700, 2)])
def test_field(fa, monkeypatch, cells, precision):
    ref = demag_field(fa, monkeypatch, cells, "double", "pad=0,fixed=0")
    h = demag_field(fa, monkeypatch, cells, precision, "")
    assert float(np.abs(h - ref).max() / np.abs(ref).max()) <= BAR[precision]
