"""One-root solves at the edges of the solver's own forms: spaces that one block holds (up to
2,048 determinants, two rows a thread beyond 1,024) with a basis of up to 16 vectors, and
mixed-precision solves whose FP32 products take each form of the single-vector product."""
import ctypes

import numpy as np
import numpy.testing as npt
import pytest
import scipy.sparse as sp

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals, spin_orbital
from tests.test_gpu_abi import Stats, eng, p  # noqa: F401

pytestmark = pytest.mark.gpu


def _dense(op):
    data, indices, indptr = op.export()
    a = sp.csr_matrix((data, indices, indptr), shape=op.shape).toarray()
    return a + np.tril(a, -1).T


def _residual(h, e, c):
    return np.linalg.norm(h @ c - e * c)


# ncv 17 and more: the basis reaches 16 columns before a restart
@pytest.mark.parametrize("ndet", [2, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049])
@pytest.mark.parametrize("ncv", [-1, 17, 24])
def test_spaces_that_one_block_holds(ndet, ncv):
    _, one, two = seeded_integrals(9, 6, 80)
    full = pyci.fullci_wfn(9, 4, 3)
    full.add_all_dets()
    dets = full.to_det_array()
    w = pyci.fullci_wfn(9, 4, 3, dets[np.random.default_rng(ndet).permutation(len(dets))[:ndet]])
    op = pyci.sparse_op(pyci.hamiltonian(0.0, one, two), w)
    es, cs = op.solve(ncv=ncv)
    h = _dense(op)
    assert abs(es[0] - np.linalg.eigvalsh(h)[0]) < 1e-10
    assert _residual(h, es[0], cs[0]) < 1e-9
    npt.assert_allclose(np.linalg.norm(cs[0]), 1.0, atol=1e-12)


# full spaces of 400 to 1,764 determinants, with and without parity sectors
@pytest.mark.parametrize("nb,nu,nd", [(6, 3, 3), (7, 3, 2), (7, 3, 3), (9, 2, 2), (9, 3, 1)])
@pytest.mark.parametrize("storage", ["csr", "direct"])
def test_small_full_spaces(nb, nu, nd, storage):
    _, one, two = seeded_integrals(nb, 6, 81)
    w = pyci.fullci_wfn(nb, nu, nd)
    w.add_all_dets()
    ham = pyci.hamiltonian(0.0, one, two)
    op = pyci.sparse_op(ham, w, storage=storage)
    es, cs = op.solve(ncv=20)
    h = _dense(pyci.sparse_op(ham, w, storage="csr"))
    assert abs(es[0] - np.linalg.eigvalsh(h)[0]) < 1e-10
    assert _residual(h, es[0], cs[0]) < 1e-9


# panels with 16 lanes and with a wave a row, ordered rows of a full space, rows without panels
# of a full space and of short ones
@pytest.mark.parametrize("kind,nb,nu,nd,ndet", [("fullci", 16, 3, 3, 19999), ("genci", 32, 5, 0, 40000),
                                                ("fullci", 10, 5, 4, 0), ("fullci", 9, 4, 4, 0), ("fullci", 20, 4, 3, 6000)])
def test_mixed_precision_over_stored_operators(eng, kind, nb, nu, nd, ndet):  # noqa: F811
    """The FP64 phase finishes what the FP32 products began: fewer FP64 products than a solve
    without them, and the same state."""
    L, ctx = eng
    _, one, two = seeded_integrals(nb if kind == "fullci" else nb // 2, 4, 82)
    if kind == "genci":
        one, two = spin_orbital(one, two)
    cls = pyci.fullci_wfn if kind == "fullci" else pyci.genci_wfn
    w = cls(nb, nu, nd)
    if ndet:
        for e in range(3):
            w.add_excited_dets(e)
        full = cls(nb, nu, nd)
        full.add_all_dets()
        rest = full.to_det_array()
        dets = np.concatenate([w.to_det_array(), rest[np.random.default_rng(ndet).permutation(len(rest))]])
        _, at = np.unique(dets.reshape(len(dets), -1), axis=0, return_index=True)
        dets = np.ascontiguousarray(dets[np.sort(at)[:ndet]])
    else:
        w.add_all_dets()
        dets = np.ascontiguousarray(w.to_det_array())
    n = len(dets)
    ham, wfn, op = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    dp, up = ctypes.c_double, ctypes.c_uint64
    assert L.pyci_ham_create(ctx, nb, 0.0, p(one, dp), p(two, dp), ctypes.byref(ham)) == 0
    assert L.pyci_wfn_create(ctx, 1 if kind == "fullci" else 2, nb, nu, nd, n, p(dets, up), ctypes.byref(wfn)) == 0
    assert L.pyci_op_create(ham, wfn, -1, -1, 1, ctypes.byref(op)) == 0
    out = []
    for precision in (0, 1):
        ev, vec, st = np.zeros(1), np.zeros(n), Stats()
        assert L.pyci_op_solve(op, 1, None, -1, -1, 1e-12, precision, p(ev, dp), p(vec, dp), ctypes.byref(st)) == 0
        y = np.zeros(n)
        assert L.pyci_op_matvec(op, 1, p(vec, dp), p(y, dp)) == 0
        assert np.linalg.norm(y - ev[0] * vec) < 1e-9
        out.append((ev[0], vec, st))
    (e64, v64, s64), (e32, v32, s32) = out
    assert abs(e64 - e32) < 1e-10
    assert s64.sigma_calls_f32 == 0 and 0 < s32.sigma_calls_f32 < s32.sigma_calls
    assert s32.sigma_calls - s32.sigma_calls_f32 < s64.sigma_calls
    L.pyci_op_destroy(op)
    L.pyci_wfn_destroy(wfn)
    L.pyci_ham_destroy(ham)
