"""Row sort of enumerated rows on both sides of the one-wave limit of 128 entries."""
import pytest

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals
from tests.test_gpu_csr import check_csr

pytestmark = pytest.mark.gpu


# rows of 2, 7, 127 and 130 entries
@pytest.mark.parametrize("nb,npair", [(2, 1), (5, 2), (45, 3), (46, 3)])
def test_doci_rows_match_oracle(oracle, nb, npair):
    _, one, two = seeded_integrals(nb, 4, 60)
    wfn = pyci.doci_wfn(nb, npair, npair)
    wfn.add_all_dets()
    ham = pyci.hamiltonian(0.0, one, two)
    check_csr(pyci.sparse_op(ham, wfn), oracle.csr_build("doci", nb, npair, npair, wfn.to_det_array(), one, two))
