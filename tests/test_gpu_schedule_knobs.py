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


# the knobs that choose between the demag routes, against the oracle (the bars
# of test_gpu_parity.py: FP64 1e-11 of the largest value, FP32 2e-6): slabs and
# their separate passes, padded and at 2n, ky classes and theirs, long z lines
@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("cells", [(32, 16, 4), (64, 32, 8), (16, 16, 6), (64, 48, 8), (13, 37, 5), (5, 160, 6),
                                   (6, 300, 3), (9, 20, 11)])
@pytest.mark.parametrize("tune", ["slab=0", "skew=0", "slab=0,pad=0", "skew=0,pad=0", "pad=0"])
def test_routes_match_oracle(fa, oracle_mod, monkeypatch, cells, precision, tune):
    monkeypatch.setenv("FULLMAG_FDM_TUNE", tune)
    nx, ny, nz = cells
    gpu = backend(fa, cells, precision)
    n = int(np.prod(cells))
    cfg = oracle_mod.OracleConfig(nx=nx, ny=ny, nz=nz, dx=4e-9, dy=3e-9, dz=2e-9, ms=8e5, a=1e-11, alpha=0.1)
    want = oracle_mod.OracleProblem(cfg, fa.generate_random_unit_vectors(17 + n, n)).observe()["h_demag"]
    bar = 1e-11 if precision == "double" else 2e-6
    np.testing.assert_allclose(gpu.copy_h_demag(), want, rtol=0, atol=bar * np.abs(want).max())
    gpu.close()
