"""CSR rows of selected sets built by testing pairs of determinants: bit for bit the
oracle's, and those of the enumerating build, which a set with one determinant of another
electron count takes, and one that holds a determinant twice."""
import numpy as np
import numpy.testing as npt
import pytest

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals, spin_orbital
from tests.test_gpu_csr import check_csr

pytestmark = pytest.mark.gpu

SPACE = {"fullci": (9, 4, 3), "genci": (18, 5, 0)}
CLS = {"fullci": pyci.fullci_wfn, "genci": pyci.genci_wfn}


def _set(kind, ndet):
    nb, nu, nd = SPACE[kind]
    _, one, two = seeded_integrals(nb if kind == "fullci" else nb // 2, 6, 50)
    if kind == "genci":
        one, two = spin_orbital(one, two)
    full = CLS[kind](nb, nu, nd)
    full.add_all_dets()
    dets = full.to_det_array().reshape(len(full), -1)
    return dets[np.random.default_rng(ndet).permutation(len(full))[:ndet]], one, two


def _wfn(kind, dets):
    return CLS[kind](*SPACE[kind], dets.reshape((-1, 2, 1) if kind == "fullci" else (-1, 1)))


# a wave's 8 rows, a chunk of 64 and a block of 4,096 columns, and their neighbours
@pytest.mark.parametrize("kind", ["fullci", "genci"])
@pytest.mark.parametrize("ndet", [1, 2, 7, 8, 9, 33, 63, 64, 65, 1000, 4095, 4096, 4097, 8250])
def test_pair_rows_match_oracle(oracle, kind, ndet):
    nb, nu, nd = SPACE[kind]
    dets, one, two = _set(kind, ndet)
    op = pyci.sparse_op(pyci.hamiltonian(0.0, one, two), _wfn(kind, dets))
    check_csr(op, oracle.csr_build(kind, nb, nu, nd, dets, one, two))
    npt.assert_array_equal(op.diagonal(), oracle.diagonal(kind, nb, nu, nd, dets, one, two))


@pytest.mark.parametrize("kind", ["fullci", "genci"])
@pytest.mark.parametrize("nrow,ncol,symmetric", [(77, 4100, False), (5000, 77, False), (4300, 4300, True)])
def test_pair_rows_of_a_part_match_oracle(oracle, kind, nrow, ncol, symmetric):
    nb, nu, nd = SPACE[kind]
    dets, one, two = _set(kind, 5000)
    op = pyci.sparse_op(pyci.hamiltonian(0.0, one, two), _wfn(kind, dets), nrow, ncol, symmetric=symmetric)
    check_csr(op, oracle.csr_build(kind, nb, nu, nd, dets, one, two, nrow=nrow, ncol=ncol, symmetric=symmetric))


@pytest.mark.parametrize("kind", ["fullci", "genci"])
def test_pair_rows_match_enumerated_rows(kind):
    dets, one, two = _set(kind, 3000)
    other = dets[:1].copy()
    other[0, 0] |= ~other[0, 0] & (other[0, 0] + np.uint64(1))  # one electron more
    ham = pyci.hamiltonian(0.0, one, two)
    a = pyci.sparse_op(ham, _wfn(kind, dets), symmetric=False)
    b = pyci.sparse_op(ham, _wfn(kind, np.concatenate([dets, other])), 3000, 3000, symmetric=False)
    for x, y in ((a.indptr(), b.indptr()), (a.indices(), b.indices()), (a.data(), b.data())):
        npt.assert_array_equal(x, y)


@pytest.mark.parametrize("kind", ["fullci", "genci"])
def test_rows_of_a_set_with_a_determinant_twice(kind):
    """The rows of a set whose last determinant is there twice: each of the two has its own
    diagonal and none of the other, the rest find one of them."""
    dets, one, two = _set(kind, 700)
    ham = pyci.hamiltonian(0.0, one, two)
    n = len(dets) - 1
    rows = []
    for d in (dets, np.concatenate([dets, dets[-1:]])):
        data, indices, indptr = pyci.sparse_op(ham, _wfn(kind, d), symmetric=False).export()
        rows.append([dict(zip(indices[a:b], data[a:b])) for a, b in zip(indptr, indptr[1:])])
        assert [len(r) for r in rows[-1]] == np.diff(indptr).tolist()
    once, twice = rows
    for r in range(n):
        expect = dict(once[r])
        if n in expect and n not in twice[r]:
            expect[n + 1] = expect.pop(n)
        assert twice[r] == expect
    last = {c: v for c, v in once[n].items() if c != n}
    assert twice[n] == {**last, n: once[n][n]} and twice[n + 1] == {**last, n + 1: once[n][n]}
