"""The XC gradients' second-derivative terms for every shell type against the oracle: SP, D and F shells in one molecule,
spherical and Cartesian, restricted and unrestricted (one and two spins' coefficients in one pass).

Tolerance: the oracle and the kernels sum the same terms in other orders (as tests/test_gpu_gradients.py)."""

import numpy as np
import pytest

import oracle
from helpers import ids, random_density
from pdynamo3_amd import basis, molecules

pytestmark = pytest.mark.gpu


def _with_f_shell(spec, z):
    """The specification with an uncontracted F shell more on element z."""
    out, p = [], 0
    while p < len(spec):
        element, shells, start = int(spec[p]), int(spec[p + 1]), p + 2
        p = start
        for _ in range(shells):
            p += 3 + int(spec[p + 2]) * (2 + int(spec[p + 1]) - int(spec[p]))
        more = [3.0, 3.0, 1.0, 0.9, 1.0] if element == z else []
        out += [spec[start - 2], shells + (1 if more else 0)] + list(spec[start:p]) + more
    return np.array(out, dtype=np.float64)


@pytest.mark.parametrize("spherical, functions", [(True, 25), (False, 29)])
def test_gradients_with_f_functions(spherical, functions):
    from pdynamo3_amd import integrator
    Z, xyz = molecules.water()
    spec = _with_f_shell(basis.element_spec(basis.load_basis("6-31g_st"), Z), 8)
    P = random_density(functions, 5, seed=11)
    g = integrator.QuadratureGrid(Z, xyz, 0)
    g.set_basis(spec, spherical, "fp64")
    assert g.number_of_functions == functions
    got, both = g.gradients(ids("blyp"), P), g.gradients_uks(ids("blyp"), 0.55 * P, 0.45 * P)
    g.close()
    ref = oracle.oracle().setup(0, Z, xyz, spec, spherical, ids("blyp"))
    assert np.max(np.abs(got - ref.gradients(P, 8))) < 1e-9
    assert np.max(np.abs(both - ref.gradients_uks(0.55 * P, 0.45 * P, 8))) < 1e-9
