"""
The panels of the blocked Householder QR (csrc/qr.hip): row counts around the sizes
at which the panel kernels change (64 .. 2048 rows), panels of fewer than 32 columns,
columns that need no reflector, wide and batched matrices. Against
numpy.linalg.qr, whose conventions the kernels follow; for matrices whose R is well
conditioned both agree to rounding (4 max(m, n) eps relative to the largest entry times the
condition number of the leading columns, bounded here by 200).
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("m", [1, 2, 31, 33, 63, 65, 100, 129, 257, 513, 700, 1025, 2049])
@pytest.mark.parametrize("n", [1, 5, 32, 33, 70])
def test_panels_match_lapack(m, n):
    rng = np.random.default_rng(m * 100 + n)
    a = orc.crandn((m, n), rng)
    a[np.arange(min(m, n)), np.arange(min(m, n))] += 4 * np.sqrt(max(m, n))
    q, r = (backend.to_host(x) for x in backend.qr(backend.as_dev(a)))
    qr, rr = np.linalg.qr(a)
    tol = 4 * max(m, n) * EPS * 200
    assert np.abs(q - qr).max() <= tol and np.abs(r - rr).max() <= tol * np.abs(rr).max()
    k = min(m, n)
    assert np.abs(q.conj().T @ q - np.eye(k)).max() < 1e-13
    assert np.abs(q @ r - a).max() <= 1e-13 * np.abs(a).max() * np.sqrt(k)


@pytest.mark.parametrize("m", [40, 130, 600, 1500, 2200])
def test_panels_without_reflectors(m):
    """Columns that are already reduced (tau = 0), zero columns and repeated ones:
    Q stays orthonormal, Q R reproduces the input, R stays upper triangular."""
    rng = np.random.default_rng(m)
    n = 37
    a = orc.crandn((m, n), rng)
    a[:, 3] = 0
    a[:, 7] = a[:, 2]
    a[1:, 0] = 0
    a[0, 0] = 2.5
    q, r = (backend.to_host(x) for x in backend.qr(backend.as_dev(a)))
    assert np.abs(q.conj().T @ q - np.eye(n)).max() < 1e-13
    assert np.abs(q @ r - a).max() <= 1e-12 * np.abs(a).max()
    assert np.all(np.tril(r, -1) == 0) and r[0, 0] == 2.5


@pytest.mark.parametrize("nb,m,n", [(5, 70, 40), (3, 300, 33), (2, 1100, 50)])
def test_batched_panels_equal_single_ones(nb, m, n):
    rng = np.random.default_rng(nb)
    a = orc.crandn((nb, m, n), rng)
    q, r = (backend.to_host(x) for x in backend.qr_batched(backend.as_dev(a)))
    for b in range(nb):
        assert np.abs(q[b].conj().T @ q[b] - np.eye(n)).max() < 1e-13
        assert np.abs(q[b] @ r[b] - a[b]).max() <= 1e-12 * np.abs(a[b]).max()
        one = backend.to_host(backend.qr(backend.as_dev(a[b]))[1])
        assert np.abs(one - r[b]).max() <= 1e-12 * np.abs(one).max()
