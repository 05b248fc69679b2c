"""XC gradients against automatic derivatives of the energy in 64 bits (perf/cases.py, which shares no code with the library)
at the atom counts where the weight terms' kernel changes its layout: 16 lanes a point (3 and 15 atoms), 32 (18), one wave
with one, two and three atoms per lane (33, 66, 129).

Tolerance: basis functions below 1e-10 at all points of a block are left out of its sums, so that a term of the gradient
is off by at most about 1e-10 times the density's and the functional's factors; the atoms' gradients are 0.1 to 1."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters", [1, 5, 6, 11, 22, 43])
def test_gradients_against_automatic_derivatives(waters):
    from perf import cases
    case = cases._case("gradients", waters, spherical=waters % 2 == 0, functional="pbe" if waters % 2 else "blyp",
                       accuracy=2 if waters < 20 else 1)
    got = cases.run(cases.prepare(case, 4))["gradients"]
    Z, xyz, _, P = cases._molecules(case, 4)[0]
    _, _, want = cases._exact_xc(case, Z, xyz, P, True)
    worst = np.max(np.abs(got - want))
    print(waters, worst, np.max(np.abs(want)))
    assert worst < 2e-8
