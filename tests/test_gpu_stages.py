"""Stages with one to five earlier slopes and the error pass on the uniform
stage kernel: every integrator on masked and unmasked grids against the oracle
(the FP64 bars of test_gpu_parity.py: max|dm| 1e-10, energies 1e-9), with the
diagnostics that an accepted adaptive step takes from its error pass."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integrator", ["heun", "rk4", "rk23", "dp45", "abm3"])
@pytest.mark.parametrize("cells", [(16, 12, 1), (70, 5, 3), (9, 6, 11)])
@pytest.mark.parametrize("masked", [False, True])
def test_integrators_match_oracle(fa, oracle_mod, integrator, cells, masked):
    nx, ny, nz = cells
    n = nx * ny * nz
    cell = (4e-9, 3e-9, 2e-9)
    mask = (np.random.default_rng(n).random(n) < 0.8).astype(np.uint8) if masked else None
    m0 = fa.generate_random_unit_vectors(31 + n, n)
    h = (2e4, -1e4, 5e3)
    gpu = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=cell, initial_magnetization=m0,
                                         saturation_magnetisation=8e5, exchange_stiffness=1.3e-11, damping=0.2,
                                         external_field=h, active_mask=mask, integrator=integrator,
                                         adaptive_max_error=1e-4, demag_kernel="device"))
    cpu = oracle_mod.OracleProblem(oracle_mod.OracleConfig(nx=nx, ny=ny, nz=nz, dx=cell[0], dy=cell[1], dz=cell[2],
                                                           ms=8e5, a=1.3e-11, alpha=0.2, h_ext=h, active_mask=mask,
                                                           integrator=integrator, max_error=1e-4), m0)
    for _ in range(6):
        g = gpu.step(5e-14)
        r = cpu.step(5e-14)
    assert float(np.abs(gpu.copy_m() - cpu.m).max()) <= 1e-10
    for key, val in (("e_ex", g.e_ex), ("e_demag", g.e_demag), ("e_total", g.e_total)):
        assert abs(val - r[key]) <= 1e-9 * max(abs(r["e_ex"]), abs(r["e_demag"]))
    assert abs(g.max_h_eff - r["max_h_eff"]) <= 1e-9 * r["max_h_eff"]
    assert abs(g.max_dm_dt - r["max_dm_dt"]) <= 1e-9 * r["max_dm_dt"]
    if integrator in ("rk23", "dp45"):
        assert abs(g.dt_suggested - r["suggested_next_dt"]) <= 1e-6 * r["suggested_next_dt"]
    gpu.close()
