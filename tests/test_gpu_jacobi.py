"""
The rounds of the block Jacobi iteration (csrc/svd.hip): column counts around the
block and pair widths, numbers of rounds around the distance between two full
rounds, and spectra that are hard for it (multiple singular values, exact rank
deficiency, columns that are zero, twelve decades). Reference: LAPACK through NumPy.
Singular values within the backward-error bound of a stable SVD, 4 q eps
sigma_max; vectors orthonormal to 1e-12; the product within 1e-11 of the input's
largest entry, as in the other split tests.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _matrix(kind, q, rng):
    if kind == "random":
        return orc.crandn((q, q), rng)
    u, _ = np.linalg.qr(orc.crandn((q, q), rng))
    v, _ = np.linalg.qr(orc.crandn((q, q), rng))
    x = np.arange(q) / max(q - 1, 1)
    s = {"graded": 10.0 ** (-12 * x), "multiple": np.where(x < 0.5, 1.0, 0.25),
         "deficient": np.where(x < 0.4, 1.0 - x, 0.0)}.get(kind, 1.0 - 0.9 * x)
    t = (u * s) @ v.conj().T
    if kind == "zero columns":
        t[:, 1::3] = 0
    return t


@pytest.mark.parametrize("q", [1, 15, 16, 17, 32, 33, 64, 127, 144, 145, 161, 290])
@pytest.mark.parametrize("kind", ["random", "graded", "multiple", "deficient", "zero columns"])
def test_split_over_the_rounds(q, kind):
    rng = np.random.default_rng(q)
    t = _matrix(kind, q, rng)
    ref = np.linalg.svd(t, compute_uv=False)
    for distr in ("left", "right"):
        a0, a1, s = backend.svd_split(backend.as_dev(t), distr, 1e-26)
        assert np.all(np.abs(s - ref) <= 4 * q * EPS * ref[0])
        a0, a1 = backend.to_host(a0), backend.to_host(a1)
        k = a0.shape[1]
        iso = a0 if distr == "right" else a1.conj().T
        assert np.abs(iso.conj().T @ iso - np.eye(k)).max() < 1e-12
        assert np.abs(a0 @ a1 - t).max() <= 1e-11 * np.abs(t).max()


@pytest.mark.parametrize("q", [144, 290])
@pytest.mark.parametrize("kind", ["random", "graded", "multiple", "zero columns"])
@pytest.mark.parametrize("precond32", [False, True])
def test_svd_with_accumulated_rotations(q, kind, precond32):
    rng = np.random.default_rng(q + 1)
    t = _matrix(kind, q, rng)
    u, s, vh = (backend.to_host(x) for x in backend.svd(backend.as_dev(t), precond32=precond32))
    ref = np.linalg.svd(t, compute_uv=False)
    assert np.all(np.abs(s - ref) <= 4 * q * EPS * ref[0])
    assert np.abs((u * s) @ vh - t).max() <= 1e-11 * np.abs(t).max()
    assert np.abs(vh @ vh.conj().T - np.eye(q)).max() < 1e-12
    k = int(np.count_nonzero(s > 1e-13 * s[0]))
    assert np.abs(u[:, :k].conj().T @ u[:, :k] - np.eye(k)).max() < 1e-12
