"""
The Jacobi phase of small matrices in one launch: column counts at the edges of its
row groups (16) and of its limits (64 columns with V, 80 without), tall and wide
matrices, spectra as in test_gpu_jacobi.py, and batches whose problems need different
numbers of sweeps. Reference: LAPACK through NumPy, tolerances of test_gpu_jacobi.py.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_jacobi import EPS, _matrix

pytestmark = pytest.mark.gpu


def _check_svd(t, u, s, vh):
    q = min(t.shape)
    ref = np.linalg.svd(t, compute_uv=False)
    assert np.all(np.abs(s - ref) <= 4 * max(t.shape) * EPS * ref[0])
    assert np.abs((u * s) @ vh - t).max() <= 1e-11 * np.abs(t).max()
    kept = s > 1e-10 * ref[0]
    assert np.abs(u[:, kept].conj().T @ u[:, kept] - np.eye(kept.sum())).max() < 1e-12
    # V is a product of rotations times an isometry (the right factor of a tall matrix)
    v = (vh if t.shape[0] >= t.shape[1] else u.conj().T)
    assert np.abs(v @ v.conj().T - np.eye(q)).max() < 1e-12


@pytest.mark.parametrize("q", [1, 2, 3, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65])
@pytest.mark.parametrize("shape", ["square", "tall", "wide"])
def test_svd_batches(q, shape):
    rng = np.random.default_rng(q)
    mats = [_matrix(k, q, rng) for k in ("random", "graded", "multiple", "deficient",
                                         "zero columns")]
    if shape != "square":
        w, _ = np.linalg.qr(orc.crandn((q + 37, q), rng))
        mats = [w @ t if shape == "tall" else t @ w.T for t in mats]
    u, s, vh, info = backend.svd_batched(backend.as_dev(np.stack(mats)), return_info=True)
    u, s, vh = (backend.to_host(x) for x in (u, s, vh))
    info = np.asarray(info.cpu() if hasattr(info, "cpu") else info).reshape(-1)
    assert info[1] == 0 and info[2] == 0 and 0 <= info[0] < 20
    for b, t in enumerate(mats):
        _check_svd(t, u[b], s[b], vh[b])


@pytest.mark.parametrize("m,n", [(47, 47), (48, 70), (49, 49), (65, 65), (90, 79), (79, 90),
                                 (80, 80), (81, 81), (5, 200), (200, 5)])
@pytest.mark.parametrize("kind", ["random", "graded", "deficient"])
def test_splits(m, n, kind):
    rng = np.random.default_rng(m * n)
    q = min(m, n)
    t = _matrix(kind, q, rng)
    w, _ = np.linalg.qr(orc.crandn((max(m, n), q), rng))
    t = w @ t if m >= n else t @ w.T
    ref = np.linalg.svd(t, compute_uv=False)
    for distr in ("left", "right"):
        a0, a1, s = backend.svd_split(backend.as_dev(t), distr, 1e-26)
        assert np.all(np.abs(s - ref) <= 4 * max(m, n) * EPS * ref[0])
        a0, a1 = backend.to_host(a0), backend.to_host(a1)
        k = a0.shape[1]
        iso = a0 if distr == "right" else a1.conj().T
        assert np.abs(iso.conj().T @ iso - np.eye(k)).max() < 1e-12
        assert np.abs(a0 @ a1 - t).max() <= 1e-11 * np.abs(t).max()
