"""compute_rdms of selected sets through pairs of determinants against the CPU oracle, and
against the enumerating kernel, which a set with one determinant of another electron
count takes."""
import numpy as np
import numpy.testing as npt
import pytest

import pyci_amd as pyci
from tests.test_gpu_csr_pairs import CLS, SPACE, _set, _wfn

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


# a wave's 8 rows, a chunk of 64 and a block of 4,096 columns, and their neighbours
@pytest.mark.parametrize("kind", ["fullci", "genci"])
@pytest.mark.parametrize("ndet", [1, 2, 8, 9, 64, 65, 700, 4096, 4097])
def test_pair_rdms_match_oracle(oracle, kind, ndet):
    dets, _, _ = _set(kind, ndet)
    c = np.random.default_rng(ndet).normal(size=ndet)
    c /= np.linalg.norm(c)
    o = oracle.rdms(kind, SPACE[kind][0], dets, c)
    # elements are sums of at most ndet products of a unit vector's entries, on both sides
    for a, b in zip(pyci.compute_rdms(_wfn(kind, dets), c), o):
        npt.assert_allclose(a, b, rtol=0, atol=2 * EPS * (ndet + 2))


@pytest.mark.parametrize("kind", ["fullci", "genci"])
def test_pair_rdms_match_enumerated_ones(kind):
    dets, _, _ = _set(kind, 3000)
    c = np.random.default_rng(1).normal(size=3001)
    c[-1] = 0.0
    c /= np.linalg.norm(c)
    other = dets[:1].copy()
    other[0, 0] |= ~other[0, 0] & (other[0, 0] + np.uint64(1))  # one electron more
    a = pyci.compute_rdms(_wfn(kind, dets), c[:-1])
    b = pyci.compute_rdms(_wfn(kind, np.concatenate([dets, other])), c)
    for x, y in zip(a, b):
        npt.assert_allclose(x, y, rtol=0, atol=2 * EPS * 3000)
    c[5] = np.nan  # reaches the same elements
    a = pyci.compute_rdms(_wfn(kind, dets), c[:-1])
    c[-1] = 0.0
    b = pyci.compute_rdms(_wfn(kind, np.concatenate([dets, other])), c)
    for x, y in zip(a, b):
        npt.assert_array_equal(np.isnan(x), np.isnan(y))


@pytest.mark.parametrize("kind", ["fullci", "genci"])
def test_rdms_of_a_set_with_a_determinant_twice(kind):
    """The same elements as by enumeration of the set (which one more determinant, of another
    electron count and without weight, takes as well)."""
    dets, _, _ = _set(kind, 700)
    dets = np.concatenate([dets, dets[-1:]])
    c = np.random.default_rng(2).normal(size=len(dets) + 1)
    c[-2], c[-1] = c[-3], 0.0
    c /= np.linalg.norm(c)
    other = dets[:1].copy()
    other[0, 0] |= ~other[0, 0] & (other[0, 0] + np.uint64(1))
    a = pyci.compute_rdms(_wfn(kind, dets), c[:-1])
    b = pyci.compute_rdms(_wfn(kind, np.concatenate([dets, other])), c)
    once = pyci.compute_rdms(_wfn(kind, dets[:-1]), c[:-2])
    for x, y in zip(a, b):
        npt.assert_allclose(x, y, rtol=0, atol=2 * EPS * 700)
    # its diagonal elements count twice
    d1 = a[0][0] if kind == "fullci" else a[0]
    o1 = once[0][0] if kind == "fullci" else once[0]
    occ = np.array([int(dets[-1, 0]) >> p & 1 for p in range(SPACE[kind][0])])
    npt.assert_allclose(np.diag(d1), np.diag(o1) + c[-2] ** 2 * occ, rtol=0, atol=2 * EPS * 700)
