"""FullCI selection and ENPT2 through sorted integral lists against the CPU oracle, which
evaluates every excitation: same determinants in the same order, same energy."""
import math

import numpy as np
import numpy.testing as npt
import pytest

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals, spin_orbital

pytestmark = pytest.mark.gpu


def _check(oracle, nb, nu, nd, count, eps_all):
    rng = np.random.default_rng(nb)
    one = rng.normal(size=(nb, nb))
    two = rng.normal(size=(nb,) * 4) * 10.0 ** rng.uniform(-4, 0, size=(nb,) * 4)  # no symmetry assumed
    strings = [[sum(1 << int(p) for p in rng.permutation(nb)[:k]) for _ in range(count)] for k in (nu, nd)]
    dets = np.unique(np.array(strings, dtype=np.uint64).T, axis=0)
    c = rng.normal(size=len(dets)) * 10.0 ** rng.uniform(-3, 0, size=len(dets))
    ham = pyci.hamiltonian(0.0, one, two)
    for eps in eps_all:
        w = pyci.fullci_wfn(nb, nu, nd, dets.reshape(-1, 2, 1))
        expect = oracle.add_hci("fullci", nb, nu, nd, dets, one, two, c, eps).reshape(-1, 2)
        e = pyci.compute_enpt2(ham, w, c, -1e3, eps=eps)
        ref, _ = oracle.enpt2("fullci", nb, nu, nd, dets, one, two, c, -1e3, eps)
        npt.assert_allclose(e, ref, rtol=1e-11)
        assert pyci.add_hci(ham, w, c, eps=eps) == len(expect)
        npt.assert_array_equal(w.to_det_array().reshape(-1, 2)[len(dets):], expect)
    return len(dets)


# no electrons or no holes of a spin, no same-spin pairs, the longest strings that are
# their own key and the first that are ranked, a list of 2,048 and the longest lists, the
# sizes around which the terms' tables need more than 64 KB of LDS
@pytest.mark.parametrize("nb,nu,nd", [(7, 3, 0), (6, 6, 3), (20, 1, 1), (32, 2, 2), (33, 2, 1), (46, 2, 1),
                                      (58, 1, 1), (59, 1, 1), (60, 1, 1), (61, 1, 1), (64, 1, 1)])
def test_fullci_lists_match_oracle(oracle, nb, nu, nd):
    _check(oracle, nb, nu, nd, 25, (0.0, 3e-3, 0.3, 1e9))


# sets large enough for sorted lists: both key forms, lists of one and two chunks, of 2,048 and
# the longest; the last set of a size that goes without and the first that sorts
@pytest.mark.parametrize("nb,nu,nd,count", [(9, 4, 3, 3000), (12, 6, 6, 300), (32, 2, 2, 400), (33, 2, 1, 600),
                                            (46, 2, 1, 700), (64, 1, 1, 5000), (16, 8, 8, 45), (16, 8, 8, 46)])
def test_sorted_lists_match_oracle(oracle, nb, nu, nd, count):
    ndet = _check(oracle, nb, nu, nd, count, (3e-3, 0.3, 1e9))
    n2, pairs = nb * nb, nb * (nb - 1) // 2
    walk = ndet * (nu * nd * n2 + (nu * (nu - 1) + nd * (nd - 1)) // 2 * pairs)
    assert (walk > 1 << 20 and 2 * walk > n2 * n2 + pairs * pairs) == (count != 45)


@pytest.mark.parametrize("kind,nb,nu,nd", [("fullci", 8, 3, 2), ("genci", 12, 4, 0)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_integrals_match_oracle(oracle, kind, nb, nu, nd, value):
    """A NaN or an infinity among the integrals decides about the excitations whose element it
    enters, and about no others."""
    rng = np.random.default_rng(nb)
    one = rng.normal(size=(nb, nb))
    two = rng.normal(size=(nb,) * 4)
    two[0, 5, 4, 5] = two[1, 2, 6, 3] = value
    strings = [[sum(1 << int(p) for p in rng.permutation(nb)[:k]) for _ in range(12)] for k in (nu, nd)]
    dets = np.unique(np.array(strings[:2 if kind == "fullci" else 1], dtype=np.uint64).T, axis=0)
    c = rng.normal(size=len(dets))
    cls = {"fullci": pyci.fullci_wfn, "genci": pyci.genci_wfn}[kind]
    ham = pyci.hamiltonian(0.0, one, two)
    for eps in (0.0, 0.1, 2.0):
        w = cls(nb, nu, nd, dets.reshape((-1, 2, 1) if kind == "fullci" else (-1, 1)))
        expect = oracle.add_hci(kind, nb, nu, nd, dets, one, two, c, eps).reshape(-1, dets.shape[1])
        assert pyci.add_hci(ham, w, c, eps=eps) == len(expect)
        npt.assert_array_equal(w.to_det_array().reshape(-1, dets.shape[1])[len(dets):], expect)


def test_rows_past_two_to_the_24():
    """Additions from the last of 17,000,000 determinants (the first of 28 spin orbitals and 11
    electrons in colex order), which are those of that determinant alone outside the set."""
    nb, nocc, ndet = 28, 11, 17_000_000
    _, one, two = seeded_integrals(nb // 2, 6, 77)
    one, two = spin_orbital(one, two)
    ham = pyci.hamiltonian(0.0, one, two)
    full = pyci.genci_wfn(nb, nocc, 0)
    full.add_all_dets()
    dets = full.to_det_array()[:ndet]
    last = pyci.genci_wfn(nb, nocc, 0, dets[-1:])
    pyci.add_hci(ham, last, np.ones(1), eps=1e-3)
    expect = last.to_det_array()[1:].ravel()
    expect = expect[[sum(math.comb(p, k + 1) for k, p in enumerate(p for p in range(nb) if int(d) >> p & 1)) >= ndet
                     for d in expect]]
    c = np.zeros(ndet)
    c[-1] = 1.0
    w = pyci.genci_wfn(nb, nocc, 0, dets)
    assert len(expect) > 0
    assert pyci.add_hci(ham, w, c, eps=1e-3) == len(expect)
    npt.assert_array_equal(w.to_det_array()[ndet:].ravel(), expect)
