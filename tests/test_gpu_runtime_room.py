"""Device memory left to the runtime (6 GB) before an SCF's integrals and dense steps, with a pretended free figure: idle
blocks of the library's cache are released first, the integrals then refuse with OutOfMemory (status 7) if there is still
less, and the dense steps go on."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOM = 6 << 30


@pytest.fixture
def free_memory():
    from pdynamo3_amd import _lib
    yield _lib.lib.xq_test_free_memory
    _lib.lib.xq_test_free_memory(-1)


def _system(waters=1):
    from helpers import cluster_system
    from pdynamo3_amd import basis
    Z, xyz, spec, _ = cluster_system(waters, 9.0 * (waters / 16.0) ** (1.0 / 3.0), 1)
    return Z, xyz, spec, basis.element_spec(basis.load_basis("dgauss-a1-dftjfit"), Z)


def _refused(call):
    with pytest.raises(Exception, match="status 7") as error:
        call()
    assert "needed by the runtime" in str(error.value)


def test_integrals_refuse_without_room(free_memory):
    from pdynamo3_amd import scf
    Z, xyz, spec, fit = _system()
    g = scf.GPUIntegrals(Z, xyz, spec, False, fit)
    want, matrix = g.one_electron(), g.fit_matrix()
    free_memory(ROOM)
    for a, b in zip(g.one_electron(), want):        # just enough
        assert np.array_equal(a, b)
    free_memory(0)
    try:
        g.one_electron()                            # releases what earlier work left idle
    except Exception:
        pass
    for call in (g.one_electron, g.fit_matrix, lambda: scf.GPUIntegrals(Z, xyz, spec, False, fit)):
        free_memory(0)
        _refused(call)
    free_memory(-1)
    for a, b in zip(g.one_electron(), want):
        assert np.array_equal(a, b)
    assert np.array_equal(g.fit_matrix(), matrix)
    g.close()


def test_idle_blocks_make_room(free_memory):
    from pdynamo3_amd import scf
    Z, xyz, spec, fit = _system()
    idle = scf.GPUIntegrals(Z, xyz, spec, False, fit)
    g = scf.GPUIntegrals(Z, xyz, spec, False, None)
    want = g.one_electron()
    idle.close()                                    # its integrals are a block of more than 64 KB
    free_memory(ROOM - 65536)
    for a, b in zip(g.one_electron(), want):
        assert np.array_equal(a, b)
    g.close()


@pytest.mark.parametrize("step", ["aufbau", "commutator"])
def test_dense_steps_release_idle_blocks_and_go_on(free_memory, step):
    from pdynamo3_amd import scf
    n = 64
    rng = np.random.default_rng(3)
    F = rng.standard_normal((n, n))
    d = scf.DeviceDenseSteps(np.eye(n), scf.pack(np.eye(n)))
    call = {"aufbau": lambda: d.aufbau(scf.pack(F + F.T), 20),
            "commutator": lambda: [d.commutator(scf.pack(F + F.T), scf.pack(F @ F.T))]}[step]
    want = call()
    Z, xyz, spec, fit = _system()
    scf.GPUIntegrals(Z, xyz, spec, False, fit).close()
    g = scf.GPUIntegrals(Z, xyz, spec, False, None)
    free_memory(0)
    for a, b in zip(call(), want):                  # nothing idle is left
        assert np.array_equal(a, b)
    free_memory(ROOM - 512)
    _refused(g.one_electron)
    d.close()
    g.close()
