"""The SCF's integral code (host build of the GPU work items, tests/native) against quadratures that share no code with it."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

from pdynamo3_amd import _lib, basis

HERE = os.path.dirname(os.path.abspath(__file__))
POWERS = ([(0, 0, 0)], [(1, 0, 0), (0, 1, 0), (0, 0, 1)],
          [(2, 0, 0), (1, 1, 0), (0, 2, 0), (1, 0, 1), (0, 1, 1), (0, 0, 2)])


@pytest.fixture(scope="module")
def host():
    subprocess.run(["make", "-s", "-C", os.path.join(HERE, "native")], check=True)
    return ctypes.CDLL(os.path.join(HERE, "native", "libqshost.so"))


def _attraction(a, A, u, b, B, v, nuclei):
    """-sum_C Z_C <x_A^u e^(-a r_A^2) | 1 / r_C | x_B^v e^(-b r_B^2)>, 1 / r = (2 / sqrt(pi)) times the integral over s of
    exp(-s^2 r^2), s^2 = p t^2 / (1 - t^2) by Gauss-Legendre, x, y and z each by Gauss-Hermite (exact)."""
    t, w = np.polynomial.legendre.leggauss(80)
    t, w = 0.5 * (t + 1.0), 0.5 * w
    h, wh = np.polynomial.hermite.hermgauss(8)
    p = a + b
    P = (a * A + b * B) / p
    s2, q = p * t ** 2 / (1.0 - t ** 2), p / (1.0 - t ** 2)
    total = 0.0
    for charge, C in nuclei:
        f = 2.0 / np.sqrt(np.pi) * w * np.sqrt(p) * (1.0 - t ** 2) ** -1.5
        for d in range(3):
            x = ((p * P[d] + s2 * C[d]) / q)[:, None] + h / np.sqrt(q)[:, None]
            f = f * np.exp(-p * s2 / q * (P[d] - C[d]) ** 2) / np.sqrt(q) * \
                np.sum(wh * (x - A[d]) ** u[d] * (x - B[d]) ** v[d], axis=1)
        total -= charge * np.sum(f)
    return total * np.exp(-a * b / p * np.sum((A - B) ** 2))


@pytest.mark.parametrize("exponent", [0.005, 0.05])
def test_attraction_of_distant_diffuse_pairs(host, exponent):
    """s, p and d functions on two atoms so far apart that the prefactor c_a c_b exp(-mu R^2) of the d pair is 1e-25.  The
    quadrature's nuclei are points, the code's Gaussians of exponent 1.3e8: 1e-10 apart at most."""
    def norm(l):
        e2, f = 2.0 * exponent, (np.pi / (2.0 * exponent)) ** 1.5
        for i in range(1, l + 1):
            f *= (2 * i - 1) / (2.0 * e2)
        return 1.0 / np.sqrt(f)

    R = np.sqrt(-np.log(1e-25 / norm(2) ** 2) * 2.0 / exponent)
    Z = np.array([8, 8], dtype=np.int32)
    xyz = np.stack([np.zeros(3), R * np.array([0.6, 0.48, 0.64])])
    shells = [{"lLow": l, "lHigh": l, "exponents": [exponent], "coefficients": [[1.0]]} for l in range(3)]
    spec = basis.element_spec({"label": "spd", "elements": {"8": {"shells": shells}}}, Z)
    S, T, V = np.zeros(210), np.zeros(210), np.zeros(210)
    assert host.qsh_one_electron(2, _lib.iptr(Z), _lib.dptr(xyz), spec.size, _lib.dptr(spec), 0, _lib.dptr(S),
                                 _lib.dptr(T), _lib.dptr(V)) == 0
    functions = [(c, u) for c in xyz for l in range(3) for u in POWERS[l]]
    nuclei = [(8.0, c) for c in xyz]
    for i in range(10, 20):
        for j in range(10):
            (A, u), (B, v) = functions[i], functions[j]
            f = 1.0
            for x in (u, v):
                f *= norm(sum(x)) * (np.sqrt(3.0) if max(x) == 1 and sum(x) == 2 else 1.0)
            want = f * _attraction(exponent, A, u, exponent, B, v, nuclei)
            got = V[i * (i + 1) // 2 + j]
            assert abs(got - want) <= 1e-8 * abs(want) + 1e-22, (u, v, got, want)


@pytest.mark.parametrize("order", range(7))
def test_boys_function_between_its_table_points(host, order):
    """Every order by the kernels' own code, at the table's points (0.05 apart), midway between them and at both sides of its
    end (T = 40), against Gauss-Legendre of t^2n exp(-T t^2) in pieces."""
    t, w = np.polynomial.legendre.leggauss(40)
    for T in (0.0, 0.025, 0.025 - 1e-12, 0.05, 1.225, 7.775, 19.975, 39.975, 40.0 - 1e-9, 40.0, 40.0 + 1e-9, 40.025, 300.0):
        F = np.zeros(order + 1)
        host.qsh_boys(order, ctypes.c_double(T), _lib.dptr(F))
        edges = np.linspace(0.0, min(1.0, 7.0 / np.sqrt(max(T, 1e-300))), 6)     # exp(-49) beyond
        for n in range(order + 1):
            want = sum(0.5 * (b - a) * np.sum(w * (0.5 * (a + b) + 0.5 * (b - a) * t) ** (2 * n) *
                                              np.exp(-T * (0.5 * (a + b) + 0.5 * (b - a) * t) ** 2))
                       for a, b in zip(edges[:-1], edges[1:]))
            assert abs(F[n] - want) <= 2e-14 * want, (T, n, F[n], want)
