"""The superblocks' tables, built on the GPU from bit masks of the functions: function counts below one word of the mask, of
whole words, and above the 64 words that one pass of the prefix sum takes.  Wrong tables would drop or displace functions in
the mixed path's V, so it is compared with the FP64 path, which does not use them.

Tolerance: the mixed path's stated one (1e-6 Eh, 1e-7 in V)."""

import numpy as np
import pytest

from helpers import ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters, functions", [(1, 19), (32, 608), (108, 2052)])
def test_mixed_equals_fp64(waters, functions):
    from pdynamo3_amd import basis, densities, integrator, molecules
    Z, xyz, rots, _ = molecules.water_cluster(waters, 14.0 * (waters / 64.0) ** (1.0 / 3.0), 5)
    spec = basis.element_spec(basis.load_basis("6-31g_st"), Z)
    P = densities.cluster_density(rots, spherical=False)
    g = integrator.QuadratureGrid(Z, molecules.to_bohr(xyz), 0)
    out = []
    for precision in ("fp64", "mixed"):
        g.set_basis(spec, False, precision)
        assert g.number_of_functions == functions
        V = np.zeros_like(P)
        out.append((g.integrate(ids("blyp"), P, V)[0], V))
    g.close()
    assert abs(out[0][0] - out[1][0]) < 1e-6
    assert np.max(np.abs(out[0][1] - out[1][1])) < 1e-7
