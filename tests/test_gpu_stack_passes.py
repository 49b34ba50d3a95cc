"""The coupled y pass and the launches shared by a stack's layers, against the
separate passes (y_split=1) and against launches by layer (per-kernel timing
on), which the other stack tests compare with the oracle: layer counts on both
sides of the coupled pass's and the packs' limits, short, ragged and long
lines, with and without a mask.

Bounds: the two routes differ by roundings of a transform of at most 1024
points and of at most 10 sources, 1e-13 of the largest field in FP64 and 2e-6
in FP32; a shared launch runs the same arithmetic per cell, so a few last bits
at most.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H_EXT = (1.5e4, -5e3, 2e3)


def make(monkeypatch, grid, layers, precision, masked, tune="", timing=False):
    import fullmag_amd as fa

    monkeypatch.setenv("FULLMAG_FDM_TUNE", tune)
    n = int(np.prod(grid))
    lps = []
    for i in range(layers):
        m0 = fa.generate_random_unit_vectors(7 * n + i, n)
        mask = None
        if masked == "all" or (masked == "some" and i == 1):
            mask = (np.random.default_rng(i).random(n) < 0.7).astype(np.uint8)
            m0[mask == 0] = 0.0
        lps.append(fa.FdmLayerPlan(magnet_name=f"L{i}", native_grid=grid, native_cell_size=(3e-9, 2.5e-9, 1e-9),
                                   native_origin=(0.0, 0.0, (2 * i + (i > 1)) * 1e-9), initial_magnetization=m0,
                                   saturation_magnetisation=(6 + i) * 1e5, exchange_stiffness=1.3e-11, damping=0.1,
                                   native_active_mask=mask))
    stack = fa.MultilayerStack(fa.FdmMultilayerPlan(common_cells=grid, convolution_cell_size=(3e-9, 2.5e-9, 1e-9),
                                                    layers=lps, external_field=H_EXT, precision=precision))
    for lay in stack.layers:
        lay.set_timing(timing)
    return stack


@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
@pytest.mark.parametrize("masked", ["none", "some", "all"])
@pytest.mark.parametrize("grid,layers", [((1, 1, 1), 2), ((5, 10, 1), 1), ((7, 3, 1), 5), ((9, 33, 1), 4),
                                         ((16, 97, 1), 3), ((33, 225, 1), 2), ((6, 257, 1), 5), ((3, 512, 1), 3),
                                         ((4, 300, 1), 4), ((2, 600, 1), 2), ((8, 12, 1), 9), ((9, 10, 2), 3)])
def test_stack_passes(monkeypatch, grid, layers, masked, precision):
    if masked == "some" and layers == 1:
        pytest.skip("one layer")
    a = make(monkeypatch, grid, layers, precision, masked)
    b = make(monkeypatch, grid, layers, precision, masked, "y_split=1", timing=True)
    ha = [lay.copy_h_demag() for lay in a.layers]
    hb = [lay.copy_h_demag() for lay in b.layers]
    scale = max(np.abs(h).max() for h in hb)
    tol = 1e-13 if precision == "double" else 2e-6
    for x, y in zip(ha, hb):
        np.testing.assert_allclose(x, y, rtol=0, atol=tol * scale)


@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
@pytest.mark.parametrize("masked", ["none", "some", "all"])
@pytest.mark.parametrize("grid,layers", [((17, 9, 1), 2), ((33, 20, 1), 4), ((12, 40, 1), 5), ((70, 33, 1), 9),
                                         ((9, 7, 3), 3)])
def test_shared_stage_launches(monkeypatch, grid, layers, masked, precision):
    a = make(monkeypatch, grid, layers, precision, masked)
    b = make(monkeypatch, grid, layers, precision, masked, timing=True)
    for dt in (1e-14, 1e-14, 2e-14):  # the last: the stored predictor is stale
        sa, sb = a.step(dt), b.step(dt)
    tol = 1e-14 if precision == "double" else 1e-6
    for x, y in zip(a.layers, b.layers):
        np.testing.assert_allclose(x.copy_m(), y.copy_m(), rtol=0, atol=tol)
    assert abs(sa.e_total - sb.e_total) <= 10 * tol * max(abs(sb.e_demag), abs(sb.e_total))
