"""The integral kernels by class of angular momenta against integrals that share no code with them (perf/cases.py: plain
torch in 64 bits): clusters whose fit shells fill less than one wave, and one wave and a part of the next, spherical and
Cartesian orbital functions; a Cartesian fit basis against the spherical one's functions of it; def2-SVP (contracted p
shells, p shells before s shells in a pair) against the host build of the same work items.

Tolerances: an integral is at most about 1e2 and a sum of some thousand rounded terms (1e-11); integrals up to 1e-12 are
stored as zero, at most about 160 of them in an element of F and 1e3 in an element of b, with coefficients below 1."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("spherical", [True, False])
@pytest.mark.parametrize("waters", [1, 4])
def test_classes_against_64_bits(waters, spherical):
    from perf import cases
    case = cases._case("integrals", waters, spherical=spherical)
    got = cases.run(cases.prepare(case, 3))
    want = cases.exact(case, 3)
    for name, tolerance in (("overlap", 1e-12), ("kinetic", 1e-11), ("nuclear", 1e-10), ("fit", 1e-10), ("fock", 1e-9),
                            ("b", 1e-8)):
        assert np.max(np.abs(got[name] - want[name])) < tolerance, name


def test_cartesian_fit_functions_contain_the_spherical_ones():
    from perf import cases
    from pdynamo3_amd import basis, densities, scf
    Z, xyz, spec, (P,) = cases._molecules(cases._case("integrals", 2), 3)[0]
    fit = basis.load_basis(cases.FIT)
    f = basis.element_spec(fit, Z)
    b = {}
    for spherical in (True, False):
        g = scf.GPUIntegrals(Z, xyz, spec, False, f, spherical)
        b[spherical] = g.fit_b(P)
        g.close()
    at = {True: 0, False: 0}
    for z in Z:
        for shell in fit["elements"][str(int(z))]["shells"]:
            for l in range(shell["lLow"], shell["lHigh"] + 1):
                T = densities.c2s(l)
                cart = b[False][at[False]:at[False] + T.shape[0]]
                assert np.max(np.abs(T.T @ cart - b[True][at[True]:at[True] + T.shape[1]])) < 1e-8
                at[True] += T.shape[1]
                at[False] += T.shape[0]
    assert at[True] == b[True].size and at[False] == b[False].size


@pytest.mark.parametrize("spherical", [True, False])
def test_def2_svp_equals_the_host_work_items(spherical):
    from perf import cases
    from pdynamo3_amd import _lib, basis, molecules, scf
    subprocess.run(["make", "-s", "-C", os.path.join(HERE, "native")], check=True)
    host = ctypes.CDLL(os.path.join(HERE, "native", "libqshost.so"))
    Z, xyz = molecules.water()
    Z, xyz = _lib.i32(Z), _lib.f64(xyz)
    spec = basis.element_spec(basis.load_basis("def2-svp"), Z)
    f = basis.element_spec(basis.load_basis(cases.FIT), Z)
    g = scf.GPUIntegrals(Z, xyz, spec, spherical, f)
    m = g.n * (g.n + 1) // 2
    want = [np.zeros(m) for _ in range(3)]
    host.qsh_one_electron(Z.size, _lib.iptr(Z), _lib.dptr(xyz), spec.size, _lib.dptr(spec), int(spherical),
                          *[_lib.dptr(x) for x in want])
    D = np.zeros((m, g.n_fit))
    host.qsh_fit_integrals(Z.size, _lib.iptr(Z), _lib.dptr(xyz), spec.size, _lib.dptr(spec), int(spherical), f.size,
                           _lib.dptr(f), 1, _lib.dptr(D))
    for x, y in zip(g.one_electron(), want):
        assert np.max(np.abs(x - y)) < 1e-11
    for k in range(g.n_fit):            # every column of the stored integrals
        F = np.zeros(m)
        g.fit_fock(np.eye(g.n_fit)[k], F)
        assert np.max(np.abs(F - D[:, k])) < 1.1e-12
    g.close()


@pytest.mark.parametrize("waters", [1, 7])
def test_cartesian_fit_matrix_contains_the_spherical_one(waters):
    """Fit functions of one launch block of the packing kernel and of one and a part; 36 products of entries up to 1e2."""
    from perf import cases
    from pdynamo3_amd import basis, densities, scf
    Z, xyz, spec, _ = cases._molecules(cases._case("integrals", waters), 3)[0]
    fit = basis.load_basis(cases.FIT)
    f = basis.element_spec(fit, Z)
    M = {}
    for spherical in (True, False):
        g = scf.GPUIntegrals(Z, xyz, spec, True, f, spherical)
        full = np.zeros((g.n_fit + 1, g.n_fit + 1))
        full[np.tril_indices(g.n_fit + 1)] = g.fit_matrix()
        M[spherical] = full + np.tril(full, -1).T
        g.close()
    T = np.zeros((M[False].shape[0], M[True].shape[0]))
    at, to = 0, 0
    for z in Z:
        for shell in fit["elements"][str(int(z))]["shells"]:
            for l in range(shell["lLow"], shell["lHigh"] + 1):
                t = densities.c2s(l)
                T[at:at + t.shape[0], to:to + t.shape[1]] = t
                at, to = at + t.shape[0], to + t.shape[1]
    T[at, to] = 1.0
    assert (at + 1, to + 1) == T.shape
    assert np.max(np.abs(T.T @ M[False] @ T - M[True])) < 1e-10
