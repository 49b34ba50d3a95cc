"""In-library Newell spectra at the edges of the near and far field.

The second differences end 40 cells out along an axis or in the radius; the
octant's rows are tabulated up to there.  Sizes on both sides of each edge,
against the oracle's spectra (same formulas on the host), to the bound of the
other spectra comparisons: 1e-11 of the largest entry.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,tf", [((1, 1, 1), True), ((40, 2, 1), True), ((41, 1, 1), False), ((42, 3, 2), False),
                                      ((2, 40, 3), False), ((3, 41, 1), True), ((2, 3, 40), False),
                                      ((3, 2, 43), False), ((29, 28, 2), False), ((24, 25, 24), False)])
def test_octant_edges(cells, tf):
    import fullmag_amd as fa
    from oracle import oracle

    got = fa.compute_newell_kernel_spectra(*cells, 3e-9, 4e-9, 2e-9, thin_film_2d=tf)
    ref = oracle.newell_spectra(*cells, 3e-9, 4e-9, 2e-9, thin_film_2d=tf)
    np.testing.assert_allclose(got, ref, rtol=0, atol=1e-11 * np.abs(ref).max())
