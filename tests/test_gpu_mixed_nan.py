"""A NaN in a density has the digits of zero in the mixed quadrature: the result is that of the density with zeros there.

Tolerance: the same integer operands; only the order of the FP64 sums into V differs from run to run."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spins", [1, 2])
@pytest.mark.parametrize("waters", [1, 3])
def test_nan_in_the_density_counts_as_zero(waters, spins):
    from helpers import cluster_system, ids
    from pdynamo3_amd import densities, integrator, molecules
    cube = 9.0 * (waters / 16.0) ** (1.0 / 3.0)
    Z, xyz, spec, _ = cluster_system(waters, cube, 7, False)
    P = densities.cluster_density(molecules.water_cluster(waters, cube, 7)[2], spherical=False) / spins
    g = integrator.QuadratureGrid(Z, xyz, 1)
    g.set_basis(spec, False, "mixed")
    places = np.random.default_rng(2).integers(0, P.size, 5)
    out = {}
    for value in (0.0, np.nan):
        Q = P.copy()
        Q[places] = value
        if spins == 1:
            V = np.zeros_like(P)
            e, n, _ = g.integrate(ids("pbe"), Q, V)
            out[value == 0.0] = np.concatenate([[e, n], V])
        else:
            Va, Vb = np.zeros_like(P), np.zeros_like(P)
            e, n, _ = g.integrate_uks(ids("pbe"), Q, P, Va, Vb)
            out[value == 0.0] = np.concatenate([[e, n], Va, Vb])
    g.close()
    assert np.all(np.isfinite(out[True]))
    assert np.max(np.abs(out[False] - out[True])) <= 1e-12
