"""The batched solver's product tiles and Rayleigh-Ritz at their edges: every pair dimension
from 16 to 128, one-root and multi-root kernels, columns short of a tile."""
import numpy as np
import pytest

import pyci_amd as pyci
from pyci_amd.synthetic import seeded_integrals

pytestmark = pytest.mark.gpu

# pair dimensions 15, 21, 36, 55, 66, 91, 105, 120, padded to 16, 32, 48, 64, 80, 96, 112, 128
SHAPES = [(5, 2, 2), (6, 3, 2), (8, 2, 2), (10, 2, 1), (11, 1, 1), (13, 2, 1), (14, 1, 1), (15, 2, 1)]


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("n", [1, 5])
def test_every_pair_dimension_matches_oracle(oracle, precision, n):
    probs, refs = [], []
    for i, (nb, nu, nd) in enumerate(SHAPES):
        _, one, two = seeded_integrals(nb, 8, 40 + i)
        probs.append((pyci.hamiltonian(0.1 * i, one, two), nu, nd))
        dets = oracle.all_dets("fullci", nb, nu, nd)
        w = oracle.lowest_eigs(oracle.csr_build("fullci", nb, nu, nd, dets, one, two), n)[0]
        refs.append(np.sort(w) + 0.1 * i)
    ev, info = pyci.batch_solve(probs, n=n, tol=1e-10, precision=precision)
    assert all(info["converged"])
    for got, ref in zip(ev, refs):
        # residuals of 1e-10 |theta| leave eigenvalues within 1e-9 of the exact ones
        np.testing.assert_allclose(np.sort(got), ref, rtol=0, atol=1e-9)
