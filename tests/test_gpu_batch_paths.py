"""Batches of equal members on every demag route, bit for bit against eager
stepping: the film's y convolution, the slab kernel, the ky classes with their
inverse lines, and the separate y lines and z convolutions (one lane per column,
or in FP64 a wavefront per component), at scheduled lengths with few and many
lanes per line."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells, precisions: film 128, 448 and 1024 points; slab to 4 and to 8 layers;
# classes of 320, 512 and 1024 points, padded and not, to 4 and to 8 layers;
# separate passes of 320, 896 and 2048 points
PATHS = [((6, 56, 1), "both"), ((9, 200, 1), "both"), ((5, 512, 1), "both"),
         ((40, 100, 3), "both"), ((16, 60, 8), "both"), ((256, 10, 4), "both"),
         ((8, 160, 6), "mixed"), ((6, 150, 2), "both"), ((5, 250, 4), "both"), ((8, 512, 8), "mixed"),
         ((6, 500, 3), "double"), ((7, 512, 2), "both"), ((12, 160, 6), "double"), ((9, 150, 5), "double"),
         ((4, 440, 8), "double"), ((4, 1024, 2), "both"), ((3, 1000, 4), "double"), ((1024, 5, 2), "both")]
CASES = [(c, p) for c, which in PATHS for p in (("mixed", "double") if which == "both" else (which,))]


@pytest.mark.parametrize("cells,precision", CASES)
def test_members_match_eager_stepping(fa, cells, precision):
    n = int(np.prod(cells))
    rng = np.random.default_rng(n)
    plans = [fa.FdmPlan(cells=cells, cell_size=(5e-9, 4e-9, 3e-9),
                        initial_magnetization=fa.generate_random_unit_vectors(11 * n + i, n),
                        saturation_magnetisation=float(rng.uniform(4e5, 1.4e6)), exchange_stiffness=1.3e-11,
                        damping=float(rng.uniform(0.01, 0.5)), external_field=tuple(rng.uniform(-2e4, 2e4, 3)),
                        precision=precision, demag_kernel="device") for i in range(3)]
    members = [fa.NativeFdmBackend(p) for p in plans]
    eager = [fa.NativeFdmBackend(p) for p in plans]
    dts = [1e-13, 7e-14, 4e-14]
    run = fa.BatchRun(members, dts, steps_per_graph=2)
    for n_steps in (3, 4):
        stats = run.run(n_steps)
        for b, e, dt, s in zip(members, eager, dts, stats):
            for _ in range(n_steps):
                r = e.step(dt)
            np.testing.assert_array_equal(b.copy_m(), e.copy_m())
            np.testing.assert_array_equal(b.copy_h_demag(), e.copy_h_demag())
            assert s.e_total == r.e_total
    run.close()
    for b in members + eager:
        b.close()
