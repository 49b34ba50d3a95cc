"""Grids whose set-up at padded transform lengths does not fit the free device
memory are transformed at 2n.  130 cells along each axis: 320 points padded, 260
at 2n; the set-up holds 2.4 GB and 1.5 GB (FP64).  Two layers on a common grid of
130 x 130 x 40: 1.9 GB and 1.3 GB.  The field is the padded plan's to the FP64
bar of the other demag tests, 1e-12 of the largest value."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


class Occupied:
    """All free device memory but `leave` bytes."""

    def __init__(self, leave):
        torch.cuda.empty_cache()
        self.held = []
        while (more := torch.cuda.mem_get_info()[0] - leave) > 64 << 20:
            self.held.append(torch.empty(more, dtype=torch.uint8, device="cuda"))

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.held.clear()
        torch.cuda.empty_cache()


def test_grid(fa):
    cells = (130, 130, 130)
    n = int(np.prod(cells))
    m = fa.generate_random_unit_vectors(3, n)
    plan = fa.FdmPlan(cells=cells, cell_size=(4e-9, 3e-9, 2e-9), initial_magnetization=m,
                      saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1, precision="double",
                      demag_kernel="device")
    gpu = fa.NativeFdmBackend(plan)
    h, held = gpu.copy_h_demag(), gpu.device_bytes()
    gpu.close()
    with Occupied(2_000_000_000):
        gpu = fa.NativeFdmBackend(plan)
        assert gpu.device_bytes() < held
        np.testing.assert_allclose(gpu.copy_h_demag(), h, rtol=0, atol=1e-12 * np.abs(h).max())
        gpu.close()


def test_stack(fa):
    grid = (130, 130, 40)
    n = int(np.prod(grid))
    cell = (4e-9, 3e-9, 2e-9)
    layers = [fa.FdmLayerPlan(magnet_name=f"L{i}", native_grid=grid, native_cell_size=cell,
                              native_origin=(0.0, 0.0, i * 90e-9),
                              initial_magnetization=fa.generate_random_unit_vectors(9 + i, n),
                              saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1) for i in range(2)]
    plan = fa.FdmMultilayerPlan(common_cells=grid, convolution_cell_size=cell, layers=layers, precision="double")
    stack = fa.MultilayerStack(plan)
    want = [lay.copy_h_demag() for lay in stack.layers]
    stack.close()
    with Occupied(1_600_000_000):
        stack = fa.MultilayerStack(plan)
        for lay, h in zip(stack.layers, want):
            np.testing.assert_allclose(lay.copy_h_demag(), h, rtol=0, atol=1e-12 * np.abs(h).max())
        stack.close()
