"""qs_fit_b and qs_fit_fock of one handle from several threads at once give what they give alone."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_b_and_fock_of_one_handle_side_by_side():
    from helpers import cluster_system
    from pdynamo3_amd import basis, scf
    Z, xyz, spec, _ = cluster_system(8, 9.0 * (8 / 16.0) ** (1.0 / 3.0), 1)
    g = scf.GPUIntegrals(Z, xyz, spec, False, basis.element_spec(basis.load_basis("dgauss-a1-dftjfit"), Z))
    rng = np.random.default_rng(5)
    m = g.n * (g.n + 1) // 2

    def fock(c):
        F = np.zeros(m)
        g.fit_fock(c, F)
        return F

    calls = [(g.fit_b, rng.standard_normal(m)) for _ in range(2)] + [(fock, rng.standard_normal(g.n_fit)) for _ in range(2)]
    want = [f(x) for f, x in calls]
    wrong = []

    def work(k):
        f, x = calls[k]
        for _ in range(100):
            if not np.array_equal(f(x), want[k]):
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    g.close()
    assert wrong == []
