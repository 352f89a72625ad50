"""Calls of several threads on wave functions of their own: density matrices, selection and
ENPT2 hold the working memory that the context keeps for the time of a call only."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import numpy.testing as npt
import pytest

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals

pytestmark = pytest.mark.gpu


def _problem(nb, nu, nd, ndet, eps):
    """What one thread does again and again; sizes differ, so that kept memory would be refilled and grown."""
    _, one, two = seeded_integrals(nb, 6, nb)
    ham = pyci.hamiltonian(0.0, one, two)
    full = pyci.fullci_wfn(nb, nu, nd)
    full.add_all_dets()
    rng = np.random.default_rng(nb)
    c = rng.normal(size=len(full))
    c /= np.linalg.norm(c)
    dets = full.to_det_array()[rng.permutation(len(full))[:ndet]]

    def run():
        part = pyci.fullci_wfn(nb, nu, nd, dets)
        r1, r2 = pyci.compute_rdms(full, c)
        s1, s2 = pyci.compute_rdms(part, c[:ndet])
        e = pyci.compute_enpt2(ham, part, c[:ndet], -30.0, eps=eps)
        pyci.add_hci(ham, part, c[:ndet], eps=eps)
        return r1, r2, s1, s2, e, part.to_det_array()

    return run


def test_threads_do_not_share_working_memory():
    problems = [_problem(9, 4, 3, 300, 1e-4), _problem(10, 4, 4, 2500, 1e-5), _problem(12, 3, 2, 40, 1e-3)]
    alone = [p() for p in problems]
    with ThreadPoolExecutor(len(problems)) as pool:
        together = list(pool.map(lambda p: [p() for _ in range(40)], problems))
    for one, many in zip(alone, together):
        for got in many:
            for a, b in zip(one[:4], got[:4]):  # sums of at most 44,100 products of a unit vector's entries
                npt.assert_allclose(a, b, rtol=0, atol=2 * np.finfo(float).eps * 44100)
            npt.assert_allclose(one[4], got[4], rtol=1e-11)
            npt.assert_array_equal(one[5], got[5])
