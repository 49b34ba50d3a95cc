"""Whole-field copies of one backend from several host threads: each thread gets
the field that it asked for, bit for bit."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(24, 20, 2), (256, 256, 4)])
@pytest.mark.parametrize("precision", ["double", "mixed", "single"])
def test_concurrent_field_copies(fa, cells, precision):
    n = int(np.prod(cells))
    gpu = fa.NativeFdmBackend(fa.FdmPlan(cells=cells, cell_size=(4e-9, 4e-9, 2e-9),
                                         initial_magnetization=fa.generate_random_unit_vectors(5, n),
                                         saturation_magnetisation=8e5, exchange_stiffness=1e-11, damping=0.1,
                                         external_field=(1e4, 0.0, 0.0), precision=precision, demag_kernel="device"))
    gpu.copy_field("H_eff")  # the observable buffers exist before the threads start
    calls = [(f, name) for f in (gpu.copy_field, gpu.copy_field_f32) for name in ("m", "H_demag", "H_ex", "H_eff")]
    want = [f(name) for f, name in calls]
    wrong = []
    start = threading.Barrier(len(calls))

    def copies(k):
        f, name = calls[k]
        start.wait()
        for _ in range(20):
            if not np.array_equal(f(name), want[k]):
                wrong.append((f.__name__, name))

    threads = [threading.Thread(target=copies, args=(k,)) for k in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    gpu.close()
