"""The single-vector products of a CSR operator (a wave per row; X staged in LDS by column
panels) against scipy's product of the exported matrix."""
import numpy as np
import numpy.testing as npt
import pytest
import scipy.sparse as sp

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals, spin_orbital

pytestmark = pytest.mark.gpu


def _check(op, symmetric, seed=0):
    data, indices, indptr = op.export()
    a = sp.csr_matrix((data, indices, indptr), shape=op.shape)
    if symmetric:
        a = a + sp.tril(a, -1).T
    x = np.random.default_rng(seed).normal(size=op.shape[1])
    row = np.diff(a.indptr).max()
    bound = abs(a) @ abs(x)  # a row's products are summed in some order on either side
    npt.assert_array_less(abs(op(x) - a @ x), 2 * row * np.finfo(float).eps * bound + 1e-300)


# one panel of 20,000 columns and its neighbours, several panels, a dense reference row
@pytest.mark.parametrize("kind,nb,nu,nd,ndet", [("fullci", 16, 3, 3, 19999), ("fullci", 16, 3, 3, 20000),
                                                ("fullci", 16, 3, 3, 20001), ("genci", 32, 5, 0, 60011),
                                                ("genci", 32, 5, 0, 40000), ("fullci", 18, 3, 3, 90001)])
def test_lds_panels(kind, nb, nu, nd, ndet):
    _, one, two = seeded_integrals(nb if kind == "fullci" else nb // 2, 4, 60)
    if kind == "genci":
        one, two = spin_orbital(one, two)
    cls = pyci.fullci_wfn if kind == "fullci" else pyci.genci_wfn
    w = cls(nb, nu, nd)
    for e in range(3):
        w.add_excited_dets(e)
    first = w.to_det_array()
    full = cls(nb, nu, nd)
    full.add_all_dets()
    rest = full.to_det_array()
    dets = np.concatenate([first, rest[np.random.default_rng(ndet).permutation(len(rest))]])
    _, at = np.unique(dets.reshape(len(dets), -1), axis=0, return_index=True)
    dets = dets[np.sort(at)[:ndet]]
    op = pyci.sparse_op(pyci.hamiltonian(0.0, one, two), cls(nb, nu, nd, dets))
    assert op.size > 1 << 19
    assert 2 * op.size - ndet > 32 * ndet * -(-ndet // 20000)  # dense enough for panels
    _check(op, True)


@pytest.mark.parametrize("nrow,ncol", [(20500, 30000), (30000, 20100), (3000, 30000)])
def test_lds_panels_of_a_part(nrow, ncol):
    _, one, two = seeded_integrals(16, 4, 61)
    full = pyci.fullci_wfn(16, 3, 3)
    full.add_all_dets()
    dets = full.to_det_array()[np.random.default_rng(1).permutation(len(full))[:30000]]
    w = pyci.fullci_wfn(16, 3, 3, dets)
    _check(pyci.sparse_op(pyci.hamiltonian(0.0, one, two), w, nrow, ncol, symmetric=False), False)


def test_rows_of_full_spaces():
    """Few short rows (DOCI), few rows and many ordered rows of a full FullCI space."""
    for cls, nb, nu, nd in ((pyci.doci_wfn, 12, 5, 5), (pyci.fullci_wfn, 6, 3, 2), (pyci.fullci_wfn, 10, 5, 4)):
        _, one, two = seeded_integrals(nb, 4, 62)
        w = cls(nb, nu, nd)
        w.add_all_dets()
        _check(pyci.sparse_op(pyci.hamiltonian(0.0, one, two), w, storage="csr"), True)


# one and several panels with 16 lanes and with a wave a row, ordered rows of a full space, one
# or two chunks a row (DOCI), rows of a small set and of a large one that the panels leave out
@pytest.mark.parametrize("kind,nb,nu,nd,ndet", [("fullci", 16, 3, 3, 19999), ("fullci", 18, 3, 3, 45000),
                                                ("genci", 32, 5, 0, 40000), ("fullci", 10, 5, 4, 0), ("doci", 12, 5, 5, 0),
                                                ("fullci", 9, 4, 3, 3000), ("genci", 44, 6, 0, 100000)])
def test_non_finite_elements_stay_in_their_rows(kind, nb, nu, nd, ndet):
    """An infinity or a NaN in x reaches the rows that hold its column and no other, and as
    itself (an infinity of a row that has no other stays one)."""
    rng = np.random.default_rng(ndet)
    cls = {"fullci": pyci.fullci_wfn, "genci": pyci.genci_wfn, "doci": pyci.doci_wfn}[kind]
    _, one, two = seeded_integrals(nb if kind != "genci" else nb // 2, 4, 63)
    if kind == "genci":
        one, two = spin_orbital(one, two)
        dets = np.unique(np.sort(rng.random((2 * ndet, nb)).argpartition(nu, axis=1)[:, :nu], axis=1), axis=0)
        dets = np.bitwise_or.reduce(np.uint64(1) << dets.astype(np.uint64), axis=1)
        w = cls(nb, nu, nd, rng.permutation(dets)[:ndet].reshape(-1, 1))
    else:
        w = cls(nb, nu, nd)
        w.add_all_dets()
        if ndet:
            w = cls(nb, nu, nd, rng.permutation(w.to_det_array())[:ndet])
    op = pyci.sparse_op(pyci.hamiltonian(0.0, one, two), w, storage="csr")
    data, indices, indptr = op.export()
    row = np.repeat(np.arange(len(indptr) - 1), np.diff(indptr))
    off = row != indices  # entries of value 0 are kept: they turn an infinity into a NaN
    a = sp.coo_matrix((np.append(data, data[off]), (np.append(row, indices[off]), np.append(indices, row[off]))),
                      shape=op.shape).tocsr()
    n = op.shape[1]
    for col in sorted({0, min(20000, n - 1), min(40000, n - 1), int(a.indices[a.indptr[7] - 1]), n - 1}):
        for value in (np.inf, np.nan):
            x = rng.normal(size=n)
            x[col] = value
            y, expect = op(x), a @ x
            npt.assert_array_equal(np.isnan(y), np.isnan(expect))
            npt.assert_array_equal(np.isinf(y), np.isinf(expect))
            assert np.isfinite(y).sum() > 0


@pytest.mark.parametrize("symmetric", [True, False])
def test_panels_after_an_update(symmetric):
    """Products after update: rows and columns appended past a panel, and a small operator
    that grows into panels."""
    _, one, two = seeded_integrals(18, 4, 64)
    ham = pyci.hamiltonian(0.0, one, two)
    full = pyci.fullci_wfn(18, 3, 3)
    full.add_all_dets()
    dets = full.to_det_array()[np.random.default_rng(3).permutation(len(full))[:61000]]
    for sizes in ((39000, 41000, 61000), (900, 30000)):
        w = pyci.fullci_wfn(18, 3, 3, dets[:sizes[0]])
        op = pyci.sparse_op(ham, w, symmetric=symmetric)
        _check(op, symmetric)
        for a, b in zip(sizes, sizes[1:]):
            more = pyci.fullci_wfn(18, 3, 3, dets[a:b])
            w.add_dets_from_wfn(more)
            op.update(ham, w)
            assert op.shape == (b, b)
            _check(op, symmetric)
