"""compute_rdms over full FullCI spaces (contractions over the coefficient matrix)
against the CPU oracle and against the general kernel, which the same state reaches
when its determinants come in another order."""
import numpy as np
import numpy.testing as npt
import pytest

import pyci_amd as pyci

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _state(nb, nu, nd):
    w = pyci.fullci_wfn(nb, nu, nd)
    w.add_all_dets()
    c = np.random.default_rng(100 * nb + 10 * nu + nd).normal(size=len(w))
    return w, c / np.linalg.norm(c)


# the smallest spaces, full and nearly full strings, tiles of 16 rows and pairs, chunks of 3 and 5 tiles, strings not a multiple of 16 or 64, very
# uneven spins, one electron or one hole of a spin
@pytest.mark.parametrize("nb,nu,nd", [(1, 1, 1), (2, 1, 1), (3, 3, 1), (4, 2, 1), (8, 3, 2), (9, 4, 3), (8, 7, 2), (8, 4, 4), (12, 3, 2), (13, 2, 2), (20, 2, 1),
                                      (11, 8, 1), (13, 7, 1), (10, 5, 5), (24, 3, 1)])
def test_full_space_rdms_match_oracle(oracle, nb, nu, nd):
    w, c = _state(nb, nu, nd)
    r1, r2 = pyci.compute_rdms(w, c)
    o1, o2 = oracle.rdms("fullci", nb, w.to_det_array(), c)
    # elements are sums of at most len(w) products of a unit vector's entries, on both sides
    atol = 2 * EPS * len(w)
    npt.assert_allclose(r1, o1, rtol=0, atol=atol)
    npt.assert_allclose(r2, o2, rtol=0, atol=atol)


@pytest.mark.parametrize("nb,nu,nd", [(8, 4, 3), (10, 5, 4)])
def test_full_space_rdms_match_general_kernel(nb, nu, nd):
    w, c = _state(nb, nu, nd)
    order = np.random.default_rng(5).permutation(len(w))
    v = pyci.fullci_wfn(nb, nu, nd, w.to_det_array()[order])
    for a, b in zip(pyci.compute_rdms(w, c), pyci.compute_rdms(v, c[order])):
        npt.assert_allclose(a, b, rtol=0, atol=2 * EPS * len(w))


def test_full_space_rdms_keep_nan_where_it_was():
    """A NaN coefficient reaches the same elements as in the general kernel."""
    w, c = _state(8, 4, 3)
    c[17] = np.nan
    order = np.arange(len(w))[::-1]
    v = pyci.fullci_wfn(8, 4, 3, w.to_det_array()[order])
    for a, b in zip(pyci.compute_rdms(w, c), pyci.compute_rdms(v, c[order])):
        npt.assert_array_equal(np.isnan(a), np.isnan(b))
