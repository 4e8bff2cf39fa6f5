"""
Deflation in the tridiagonal eigensolver of the local solves (csrc/krylov.hip
tridiag_coefs): a coupling e_k is dropped when |e_k| <= eps (|d_k| + |d_{k+1}|), the last
one too. Operators with a zero on the diagonal next to 1e5 and couplings of 2^-40 = 9e-13 (a power
of two: the Lanczos vectors are unit vectors without rounding), above the breakdown
threshold and below eps 1e5 = 2e-11: the matrix counts as diagonal, so the lowest Ritz
pair is the zero and its unit vector exactly.
"""

import numpy as np
import pytest

from pytenet_amd import backend, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("diag", [(0.0, 1e5), (2e5, 0.0, 1e5), (1e5, 0.0), (3e5, 2e5, 0.0, 1e5)])
def test_last_coupling_is_dropped_against_both_neighbours(diag):
    n, k = len(diag), diag.index(0.0)
    h = np.diag(diag) + 2.0**-40 * (np.eye(n, k=1) + np.eye(n, k=-1))
    v = np.zeros((n, 1))
    v[0, 0] = 1.0
    out, energy, info = backend.krylov_local(_lib.PTN_OP_BOND, v, h.reshape(n, 1, n), None,
                                             np.ones((1, 1, 1)), n, "eigh")
    assert list(backend.to_host(info)) == [n, 0, 0, 0]
    want = np.zeros((n, 1))
    want[k, 0] = 1.0
    assert float(energy.item()) == 0.0
    assert np.array_equal(backend.to_host(out), want)
