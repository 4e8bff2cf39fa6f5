"""
The one-launch pieces of small QR factorisations (csrc/qr.hip): entry counts around
the limit of the one-workgroup copy (8192) with entries outside the range that is
factored unscaled, and the fused block update around its row limits (256; 512 in a
batch), column groups of 8 and reflector counts around 16 and 32. Reference and tolerances:
test_gpu_qr_panels.py.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_qr_panels import EPS

pytestmark = pytest.mark.gpu


def _check(a, q, r):
    k = min(a.shape)
    qr, rr = np.linalg.qr(a)
    tol = 4 * max(a.shape) * EPS * 200
    assert np.abs(q - qr).max() <= tol and np.abs(r - rr).max() <= tol * np.abs(rr).max()
    assert np.abs(q.conj().T @ q - np.eye(k)).max() < 1e-13


def _matrix(rng, m, n):
    a = orc.crandn((m, n), rng)
    a[np.arange(min(m, n)), np.arange(min(m, n))] += 4 * np.sqrt(max(m, n))
    return a


@pytest.mark.parametrize("m,n", [(3, 2), (64, 128), (128, 64), (91, 90), (91, 91), (256, 32),
                                 (257, 32)])
@pytest.mark.parametrize("scale", [1.0, 1e-280, 1e200])
def test_scaled_copies(m, n, scale):
    rng = np.random.default_rng(m + n)
    a = _matrix(rng, m, n)
    q, r = (backend.to_host(x) for x in backend.qr(backend.as_dev(a * scale)))
    _check(a, q, r / scale)


@pytest.mark.parametrize("m,n", [(33, 41), (48, 49), (64, 65), (255, 70), (256, 47), (287, 81),
                                 (289, 48), (20, 100), (16, 17)])
def test_block_updates(m, n):
    rng = np.random.default_rng(m * n)
    a = _matrix(rng, m, n)
    _check(a, *(backend.to_host(x) for x in backend.qr(backend.as_dev(a))))


@pytest.mark.parametrize("nb,m,n", [(3, 64, 47), (2, 512, 40), (2, 545, 66), (3, 30, 75)])
def test_block_updates_of_batches(nb, m, n):
    rng = np.random.default_rng(m + n)
    a = np.stack([_matrix(rng, m, n) for _ in range(nb)])
    q, r = (backend.to_host(x) for x in backend.qr_batched(backend.as_dev(a)))
    for b in range(nb):
        _check(a[b], q[b], r[b])
