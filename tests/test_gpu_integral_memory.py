"""Integrals of molecules whose pair records do not fit in one slice: the device memory a call takes beside its results, and
values that do not depend on where the slices are cut (the atoms in reverse order, whose pairs fall into other slices).
Electron-fit integrals that one launch cannot hold, against their closed form."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GB = 1 << 30


def _free():
    """Free device memory as the runtime that this library is linked with sees it (torch may have brought another)."""
    with open("/proc/self/maps") as maps:
        paths = sorted({line.split()[-1] for line in maps if "libamdhip64" in line})
    for path in paths:
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        if ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0:
            return free.value
    raise AssertionError("no runtime with a device among {}".format(paths))


def _lattice(waters):
    """Waters 6 bohr apart on a cubic lattice, each turned a little against the one before."""
    from pdynamo3_amd import molecules
    Z, xyz = molecules.water()
    Z, xyz = np.asarray(Z, dtype=np.int32), np.asarray(xyz).reshape(-1, 3)
    side, out = int(np.ceil(waters ** (1.0 / 3.0))), []
    for k in range(waters):
        c, s = np.cos(0.37 * k), np.sin(0.37 * k)
        turn = np.array([[c, -s, 0.0], [s, c, 0.0], [0.0, 0.0, 1.0]])
        out.append(xyz @ turn.T + 6.0 * np.array([k % side, k // side % side, k // side ** 2]))
    return np.tile(Z, waters), np.concatenate(out)


def _functions(Z, spec_of):
    return np.array([spec_of[int(z)] for z in Z])


def _reversed_places(Z, per_element):
    """Places of the functions, in the order of the reversed atoms."""
    first = np.concatenate([[0], np.cumsum(_functions(Z, per_element))])
    return np.concatenate([np.arange(first[a], first[a + 1]) for a in range(Z.size - 1, -1, -1)])


def _dense(packed, n):
    out = np.zeros((n, n))
    out[np.tril_indices(n)] = packed
    return out + np.tril(out, -1).T


def test_one_electron_of_300_waters():
    from pdynamo3_amd import basis, scf
    Z, xyz = _lattice(300)
    data = basis.load_basis()
    spec = basis.element_spec(data, Z)
    g = scf.GPUIntegrals(Z, xyz, spec, False, None)
    before = _free()
    got = g.one_electron()
    taken = before - _free()
    n = g.n
    g.close()
    print("functions", n, "device memory taken", taken / GB)
    assert taken < 1.2 * GB                     # S, T and V are 0.4 GB
    places = _reversed_places(Z, {z: basis.number_of_functions(data, np.array([z], dtype=np.int32), False) for z in (1, 8)})
    g = scf.GPUIntegrals(Z[::-1].copy(), xyz[::-1].copy(), spec, False, None)
    other = g.one_electron()
    g.close()
    for a, b in zip(got, other):
        A = _dense(a, n)[np.ix_(places, places)]
        assert np.max(np.abs(A - _dense(b, n))) <= 1e-12 * np.max(np.abs(A))


def test_fit_matrix_of_250_waters():
    """One tight s function per atom as the orbital basis: the fit integrals themselves stay small."""
    from pdynamo3_amd import basis, scf
    Z, xyz = _lattice(250)
    shell = {"lLow": 0, "lHigh": 0, "exponents": [50.0], "coefficients": [[1.0]]}
    spec = basis.element_spec({"label": "s", "elements": {z: {"shells": [shell]} for z in ("1", "8")}}, Z)
    data = basis.load_basis("dgauss-a1-dftjfit")
    fit = basis.element_spec(data, Z)
    g = scf.GPUIntegrals(Z, xyz, spec, False, fit)
    before = _free()
    got = g.fit_matrix()
    taken = before - _free()
    n = g.n_fit
    g.close()
    print("fit functions", n, "device memory taken", taken / GB)
    assert taken < 0.75 * GB                    # the packed matrix is 0.4 GB
    places = _reversed_places(Z, {z: basis.number_of_functions(data, np.array([z], dtype=np.int32), True) for z in (1, 8)})
    places = np.concatenate([places, [n]])
    g = scf.GPUIntegrals(Z[::-1].copy(), xyz[::-1].copy(), spec, False, fit)
    other = g.fit_matrix()
    g.close()
    A = _dense(got, n + 1)
    A = A[np.ix_(places, places)]
    B = _dense(other, n + 1)
    assert np.max(np.abs(A - B)) <= 1e-12 * np.max(np.abs(A))


def test_fit_integrals_beyond_one_launch():
    """One s function on each of 11,700 H atoms and one s fit function on an O atom: 68 million shell pairs, a wave each.
    (ab|c) = 2 pi^(5/2) / (p g sqrt(p + g)) c_a c_b c_c exp(-a R^2 / 2) F_0(T), p = 2 a, T = p g / (p + g) |P - C|^2."""
    from scipy.special import erf
    from pdynamo3_amd import basis, scf
    n, a, g = 11700, 0.1, 1.0
    rng = np.random.default_rng(8)
    xyz = np.concatenate([np.zeros((1, 3)), rng.uniform(-4.0, 4.0, (n, 3))])
    Z = np.array([8] + [1] * n, dtype=np.int32)

    def spec(on, exponent):
        shell = {"lLow": 0, "lHigh": 0, "exponents": [exponent], "coefficients": [[1.0]]}
        return basis.element_spec({"label": "s", "elements": {z: {"shells": [shell] if z == on else []} for z in ("1", "8")}}, Z)

    ints = scf.GPUIntegrals(Z, xyz, spec("1", a), False, spec("8", g))
    pairs = n * (n + 1) // 2
    assert ints.n_fit == 1 and ints.stats()["fit_rows"] == pairs > 1 << 26
    F = np.zeros(pairs)
    ints.fit_fock(np.ones(1), F)
    ints.close()
    k = np.concatenate([rng.integers(0, pairs, 200000), np.arange(1000), pairs - 1 - np.arange(1000),
                        (1 << 25) + np.arange(-500, 500), (1 << 26) + np.arange(-500, 500)])
    i = ((np.sqrt(8.0 * k + 1.0) - 1.0) / 2.0).astype(np.int64)
    i += (i + 1) * (i + 2) // 2 <= k
    i -= i * (i + 1) // 2 > k
    j = k - i * (i + 1) // 2
    assert np.all((0 <= j) & (j <= i))
    A, B = xyz[1 + i], xyz[1 + j]
    p, norm = 2.0 * a, (2.0 * a / np.pi) ** 1.5 * (2.0 * g / np.pi) ** 0.75
    T = p * g / (p + g) * np.sum((0.5 * (A + B)) ** 2, axis=1)
    F0 = 0.5 * np.sqrt(np.pi / T) * erf(np.sqrt(T))
    want = norm * 2.0 * np.pi ** 2.5 / (p * g * np.sqrt(p + g)) * np.exp(-0.5 * a * np.sum((A - B) ** 2, axis=1)) * F0
    assert np.max(np.abs(F[k] - want)) < 1e-12
