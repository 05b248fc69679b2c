"""Grid weights and weight gradients where a lane holds several atoms (3, 4, 6, 10, 16 and 24 of them), on dense lattices of C
and H atoms:

- the weights of points of the first, middle and last atoms against Becke's cell functions in numpy, all atoms against all:
  the weight of a point alone on its atom (a one-atom grid of the element) times its share of the cells.  Tolerance: a
  share of a sum of up to 1,489 products of as many factors, 1e-16 each: 1e-12;
- the XC gradients of single atoms against differences of E_xc (four points, 2e-3 bohr apart).  Tolerance: the steps'
  fourth-order error, 1.6e-11 / 30 times the fifth derivative (1e3 for the exponents here), is 6e-10, the rounding of an
  energy of 1e2 or functions that enter and leave blocks at 1e-8 a density's 1e-8 away, 1e-13 / 1e-3; 2e-8 in all."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RADIUS = {1: 0.35, 6: 0.70}         # Bragg's, Angstrom (DFTGrid.c:29-40)


def _lattice(n):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1.0 / 3.0)))
    xyz = 3.0 * np.array([[k % side, k // side % side, k // side ** 2] for k in range(n)], dtype=float)
    return np.where(np.arange(n) % 3 == 0, 6, 1).astype(np.int32), xyz + rng.uniform(-0.4, 0.4, (n, 3))


def _cells(Z, xyz, point, pairs):
    """Becke's cell products at a point, all atoms against all; the cell function is the integral of (1 - x^2)^10."""
    inverse, shift = pairs
    r = np.linalg.norm(xyz - point, axis=1)
    mu = (r[:, None] - r[None, :]) * inverse
    nu = mu + shift * (1.0 - mu * mu)
    t = np.arange(11)
    binomial = np.array([1, 10, 45, 120, 210, 252, 210, 120, 45, 10, 1], dtype=float)
    c = binomial * (-1.0) ** t / (2 * t + 1)
    poly = np.zeros_like(nu)
    for k in c[::-1]:
        poly = poly * nu * nu + k
    s = 0.5 - 0.5 / np.sum(c) * poly * nu
    np.fill_diagonal(s, 1.0)
    return np.prod(s, axis=1)


def _pairs(Z, xyz):
    d = np.linalg.norm(xyz[:, None] - xyz[None], axis=2)
    np.fill_diagonal(d, 1.0)
    radius = np.array([RADIUS[int(z)] for z in Z])
    chi = radius[:, None] / radius[None, :]
    u = (chi - 1.0) / (chi + 1.0)
    return 1.0 / d, np.clip(u / (u * u - 1.0), -0.5, 0.5)


@pytest.mark.parametrize("n", [150, 220, 300, 500, 800, 1489])
def test_weights_equal_all_pairs(n):
    from pdynamo3_amd import integrator
    Z, xyz = _lattice(n)
    alone = {}
    for z in (1, 6):
        g = integrator.QuadratureGrid([z], np.zeros((1, 3)), 0)
        alone[z] = g.points()[0]
        g.close()
    g = integrator.QuadratureGrid(Z, xyz, 0)
    points, atom, count = g.points()
    g.close()
    owner = np.repeat(atom, count)
    pairs = _pairs(Z, xyz)
    rng, checked = np.random.default_rng(1), 0
    for a in (0, 1, n // 2, n // 2 + 1, n - 2, n - 1):
        own = points[owner == a]
        for p in own[rng.integers(0, own.shape[0], 8)]:
            d = np.linalg.norm(alone[int(Z[a])][:, :3] - (p[:3] - xyz[a]), axis=1)
            k = np.argmin(d)
            assert d[k] < 1e-9
            cell = _cells(Z, xyz, p[:3], pairs)
            base = alone[int(Z[a])][k, 3]
            assert abs(p[3] - base * cell[a] / np.sum(cell)) <= 1e-12 * abs(base)
            checked += 1
    assert checked == 48


@pytest.mark.parametrize("n", [150, 220, 300, 500, 800])
def test_gradients_equal_differences(n):
    from helpers import ids, packed
    from pdynamo3_amd import basis, integrator
    Z, xyz = _lattice(n)
    shell = lambda e, l: {"lLow": l, "lHigh": l, "exponents": [e], "coefficients": [[1.0]]}
    spec = basis.element_spec({"label": "sp", "elements": {"1": {"shells": [shell(0.8, 0)]},
                                                           "6": {"shells": [shell(1.2, 0), shell(0.9, 1)]}}}, Z)
    functional = ids("pbe")

    def grid(x):
        g = integrator.QuadratureGrid(Z, x, 0)
        g.set_basis(spec, True, "fp64")
        return g

    g = grid(xyz)
    m = g.number_of_functions
    rng = np.random.default_rng(3)
    P = np.diag(rng.uniform(0.5, 1.5, m))
    P[np.arange(1, m), np.arange(m - 1)] = 0.2
    P = packed(P)
    G = g.gradients(functional, P)
    g.close()

    def energy(a, x, step):
        moved = xyz.copy()
        moved[a, x] += step
        g = grid(moved)
        e = g.integrate(functional, P)[0]
        g.close()
        return e

    h = 2e-3
    for a, x in ((0, 0), (n // 2 + 1, 1), (n - 1, 2)):
        slope = (8.0 * (energy(a, x, h) - energy(a, x, -h)) - (energy(a, x, 2 * h) - energy(a, x, -2 * h))) / (12.0 * h)
        print(n, a, G[a, x], slope - G[a, x])
        assert abs(slope - G[a, x]) <= 2e-8
