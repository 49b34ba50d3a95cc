"""Values of the schedule knobs at and beyond the edges of their ranges: the
demag field is the default schedule's to the rounding of the transforms (FP64
1e-12 and FP32 2e-6 of the largest value, the bars of the other demag tests)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BAR = {"double": 1e-12, "mixed": 2e-6}


def backend(fa, cells, precision):
    n = int(np.prod(cells))
    return fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(4e-9, 3e-9, 2e-9),
                                          initial_magnetization=fa.generate_random_unit_vectors(17 + n, n),
                                          saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                          precision=precision, demag_kernel="device"))


# scheduled x lengths (64, 28 and 1024 points) and a runtime plan (fixed=0)
@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("cells,more", [((32, 9, 1), ""), ((13, 7, 3), ""), ((500, 5, 2), ""), ((32, 9, 1), ",fixed=0")])
@pytest.mark.parametrize("rows", [-1, 1, 2, 3, 6, 24, 64, 1000])
def test_rows_per_x_workgroup(fa, monkeypatch, rows, cells, more, precision):
    monkeypatch.setenv("FULLMAG_FDM_TUNE", "")
    gpu = backend(fa, cells, precision)
    h = gpu.copy_h_demag()
    bar = BAR[precision] * np.abs(h).max()
    tune = f"x_rows={rows}{more}"
    gpu.upload_magnetization(np.zeros((int(np.prod(cells)), 3)))
    gpu.refresh_observables()  # a launch that does not run would leave this zero field
    gpu.set_schedule(tune)
    gpu.upload_magnetization(fa.generate_random_unit_vectors(17 + int(np.prod(cells)), int(np.prod(cells))))
    gpu.refresh_observables()
    assert np.abs(gpu.copy_h_demag() - h).max() <= bar
    gpu.close()
    monkeypatch.setenv("FULLMAG_FDM_TUNE", tune)
    gpu = backend(fa, cells, precision)
    assert np.abs(gpu.copy_h_demag() - h).max() <= bar
    gpu.close()


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("slab", [-1, 0, 1, 160])
def test_slab_kernel_by_its_knob(fa, monkeypatch, slab, precision):
    """The slab kernel runs where its 17 KB (FP64: 34) fit the knob's KB; 0 and
    below turn it off."""
    monkeypatch.setenv("FULLMAG_FDM_TUNE", "skew=0")
    gpu = backend(fa, (40, 100, 3), precision)
    h = gpu.copy_h_demag()
    gpu.set_schedule(f"slab={slab}")
    gpu.set_timing(True)
    gpu.refresh_observables()
    gpu.step(1e-14)
    assert ("demag_yz_slab" in gpu.timings()) == (slab == 160)
    gpu.upload_magnetization(fa.generate_random_unit_vectors(17 + 12000, 12000))
    gpu.refresh_observables()
    assert np.abs(gpu.copy_h_demag() - h).max() <= BAR[precision] * np.abs(h).max()
    gpu.close()
