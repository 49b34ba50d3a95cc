"""The scheduled transform lengths (2^a, and 10, 12 or 14 times 2 .. 64): the
demag field against the general path, which transforms at 2n with runtime
plans in FP64 (itself checked against the oracle in test_gpu_parity.py), for
the cell counts at both ends of the range that each length serves (the library
pads n cells to the next scheduled length of at least 2n)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 2n equal to a scheduled length, and the smallest n that each length serves
COUNTS = [10, 11, 12, 13, 14, 17, 20, 23, 24, 25, 28, 29, 33, 40, 41, 48, 49, 56, 57, 65, 80, 81, 96, 97, 112, 113,
          129, 160, 161, 192, 193, 224, 225, 257, 320, 321, 384, 385, 448, 449]
# each count once along x and once along y
PAIRS = list(zip(COUNTS, COUNTS[::-1]))


def demag_field(fa, monkeypatch, cells, precision, tune, mask):
    monkeypatch.setenv("FULLMAG_FDM_TUNE", tune)
    n = int(np.prod(cells))
    gpu = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(4e-9, 3e-9, 2e-9),
                                         initial_magnetization=fa.generate_random_unit_vectors(71 + n, n),
                                         saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                         enable_exchange=False, precision=precision, active_mask=mask,
                                         demag_kernel="device"))
    h = gpu.copy_h_demag()
    gpu.close()
    return h


def field_error(fa, monkeypatch, cells, precision, mask=None, tune=""):
    ref = demag_field(fa, monkeypatch, cells, "double", "pad=0,fixed=0", mask)
    h = demag_field(fa, monkeypatch, cells, precision, tune, mask)
    return float(np.abs(h - ref).max() / np.abs(ref).max())


# the FP64 field bar of the other demag tests; FP32 transforms: 2e-6
BAR = {"double": 1e-12, "mixed": 2e-6}


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("nz", [1, 2])
@pytest.mark.parametrize("nx,ny", PAIRS)
def test_x_and_y_lengths(fa, monkeypatch, nx, ny, nz, precision):
    assert field_error(fa, monkeypatch, (nx, ny, nz), precision) <= BAR[precision]


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("nz", [n for n in COUNTS if n <= 129])
def test_z_lengths(fa, monkeypatch, nz, precision):
    assert field_error(fa, monkeypatch, (5, 7, nz), precision) <= BAR[precision]


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("cells", [(33, 49, 1), (25, 17, 3), (13, 11, 11)])
def test_masked(fa, monkeypatch, cells, precision):
    mask = (np.random.default_rng(3).random(int(np.prod(cells))) < 0.8).astype(np.uint8)
    assert field_error(fa, monkeypatch, cells, precision, mask) <= BAR[precision]


@pytest.mark.parametrize("cells", [(33, 25, 1), (41, 49, 4), (17, 13, 20)])
def test_unpadded_schedule_agrees(fa, monkeypatch, cells):
    """pad=0 keeps the transforms at 2n."""
    assert field_error(fa, monkeypatch, cells, "double", tune="pad=0") <= BAR["double"]


# y and z passes in one slab kernel: every layer count, y lengths of 2, 16 and
# 32 lanes per line, whole and partial rounds of columns
@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
@pytest.mark.parametrize("nz", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("nx,ny", [(5, 13), (17, 10), (9, 100), (12, 160), (7, 256)])
def test_slab_and_separate_passes(fa, monkeypatch, nx, ny, nz, precision):
    for tune in ("", "slab=0"):
        assert field_error(fa, monkeypatch, (nx, ny, nz), precision, tune=tune) <= BAR.get(precision, 2e-6)


# ky classes of a slab: every layer count, P = 80, 160, 192, 224 and 256 entries
# per class, ny at, below and far below half the padded length
@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("nz", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("nx,ny", [(5, 149), (9, 320), (6, 384), (11, 385), (4, 449), (7, 512)])
def test_class_and_separate_passes(fa, monkeypatch, nx, ny, nz, precision):
    for tune in ("", "slab=0"):
        assert field_error(fa, monkeypatch, (nx, ny, nz), precision, tune=tune) <= BAR[precision]


@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
def test_classes_off_at_run_time(fa, precision):
    """The tensor keeps its class order when a schedule turns the classes off."""
    cells = (6, 300, 3)
    n = int(np.prod(cells))
    gpu = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(4e-9, 3e-9, 2e-9),
                                         initial_magnetization=fa.generate_random_unit_vectors(7, n),
                                         saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                         precision=precision, demag_kernel="device"))
    h = gpu.copy_h_demag()
    for tune in ("slab=0", "fixed=0", "slab=160"):
        gpu.set_schedule(tune)
        gpu.refresh_observables()
        assert np.abs(gpu.copy_h_demag() - h).max() <= BAR.get(precision, 2e-6) * np.abs(h).max()
    gpu.close()


# x frequencies k + 1/2 (slab plans) and integer ones
@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
@pytest.mark.parametrize("cells", [(5, 13, 2), (33, 17, 5), (40, 100, 3), (256, 250, 8), (256, 256, 4), (512, 100, 7),
                                   (12, 150, 6), (20, 256, 5), (256, 300, 8), (250, 149, 3)])
def test_skewed_x_frequencies(fa, monkeypatch, cells, precision):
    n = int(np.prod(cells))
    mask = (np.random.default_rng(5).random(n) < 0.8).astype(np.uint8) if cells[0] == 33 else None
    for tune in ("", "skew=0", "fixed=0"):
        assert field_error(fa, monkeypatch, cells, precision, mask, tune=tune) <= BAR.get(precision, 2e-6)
