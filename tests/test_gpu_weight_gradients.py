"""XC gradients against the oracle at the atom counts where the weight terms' kernel changes its layout: 16 lanes a point (3 and
15 atoms), 32 (18 and 30), one wave with one and two atoms per lane (33 and 66).  The grids are the smallest (VeryLow).

Tolerance: the oracle and the kernel sum the same terms in other orders (as tests/test_gpu_gradients.py)."""

import numpy as np
import pytest

import oracle
from helpers import cluster_system, ids
from pdynamo3_amd import densities, molecules

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters", [1, 5, 6, 10, 11, 22])
def test_gradients_equal_the_oracle(waters):
    from pdynamo3_amd import integrator
    cube, spherical = 9.0 * (waters / 16.0) ** (1.0 / 3.0), waters % 2 == 0
    Z, xyz, spec, _ = cluster_system(waters, cube, 7, spherical)
    P = densities.cluster_density(molecules.water_cluster(waters, cube, 7)[2], spherical=spherical)
    functional = ids("pbe" if waters % 2 else "blyp")
    g = integrator.QuadratureGrid(Z, xyz, 0)
    g.set_basis(spec, spherical, "fp64")
    got = g.gradients(functional, P)
    g.close()
    want = oracle.oracle().setup(0, Z, xyz, spec, spherical, functional).gradients(P, 8)
    worst = np.max(np.abs(got - want))
    print(waters, worst)
    assert worst < 1e-9
