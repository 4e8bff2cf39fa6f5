"""
The forms of the local solves: the whole solve of a small problem in one launch,
one-workgroup Lanczos steps on short vectors, the exponential of the tridiagonal
matrix by Taylor steps and by eigendecomposition, and the status words. Against
the oracle's Lanczos (pytenet/krylov.py) and, for the small problems, against the
launches per step (taken by the tile-mask products). The recurrence amplifies
rounding differences of the matvecs (1e-15) by the ratio of neighbouring betas; 1e-11
of the norm for up to 12 steps as in the other solver tests. Energies: 1e-12 of |H|.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend, _lib

pytestmark = pytest.mark.gpu


def _herm(rng, D, M):
    x = orc.crandn((M, D, D), rng) / np.sqrt(D)
    return np.ascontiguousarray(np.transpose(x + np.conj(np.transpose(x, (0, 2, 1))), (1, 0, 2)))


def _operator(rng, Dl, d, Dr, Ml, Mr, density=0.4):
    """Hermitian local operator: every L[:, m, :], W[m, :, :, m'], R[:, m', :] Hermitian;
    W has empty rows and single entries."""
    w = orc.crandn((Ml, d, d, Mr), rng)
    w = w + np.conj(np.transpose(w, (0, 2, 1, 3)))
    keep = rng.uniform(size=(Ml, Mr)) < density
    keep[0, 0] = True
    w = w * keep[:, None, None, :]
    return _herm(rng, Dl, Ml), w, _herm(rng, Dr, Mr)


def _solve(kind, v, l, w, r, numiter, mode, dt=0.0, **kw):
    out, en, info = backend.krylov_local(kind, v, l, w, r, numiter, mode, dt, **kw)
    return (backend.to_host(out), None if en is None else float(en[0]),
            info.cpu().numpy())


def _names(fn):
    backend.timing_begin()
    res = fn()
    return res, [x["name"] for x in backend.timing_end()]


HEFF = [(1, 1, 1, 1, 1), (1, 2, 3, 2, 3), (2, 4, 1, 5, 1), (7, 2, 9, 3, 3), (8, 4, 8, 5, 5),
        (15, 2, 17, 3, 4), (16, 2, 16, 5, 5), (17, 3, 13, 2, 5), (13, 4, 15, 5, 4),
        (16, 2, 32, 3, 3), (8, 8, 6, 4, 4), (5, 4, 31, 8, 3)]


@pytest.mark.parametrize("dims", HEFF)
@pytest.mark.parametrize("numiter", [1, 2, 11])
def test_small_heff_solves(dims, numiter):
    rng = np.random.default_rng(sum(dims) * 13 + numiter)
    Dl, d, Dr, Ml, Mr = dims
    l, w, r = _operator(rng, *dims)
    v = orc.crandn((Dl, d, Dr), rng)
    numiter = min(numiter, v.size)
    hfun = lambda x: orc.apply_local_hamiltonian(x.reshape(v.shape), w, l, r).reshape(-1)
    dt = 0.05 - 0.11j
    (got, _, info), names = _names(
        lambda: _solve(_lib.PTN_OP_HEFF, v, l, w, r, numiter, "expm", dt))
    assert "k_lz_solve" in names, names
    assert list(info) == [numiter, 0, 0, 0]
    steps, _, _ = _solve(_lib.PTN_OP_HEFF, v, l, w, r, numiter, "expm", dt, block_sparse=True)
    ref = orc.expm_krylov(hfun, v.reshape(-1), dt, numiter, hermitian=True).reshape(v.shape)
    nrm = np.linalg.norm(ref)
    assert np.linalg.norm(got - ref) < 1e-11 * nrm
    assert np.linalg.norm(got - steps) < 1e-11 * nrm
    _, en, _ = _solve(_lib.PTN_OP_HEFF, v, l, w, r, numiter, "eigh")
    eref, _ = orc.eigh_krylov(hfun, v.reshape(-1), numiter, 1)
    scale = max(1.0, abs(float(eref[0])), np.abs(hfun(v.reshape(-1))).max())
    assert abs(en - float(eref[0])) < 1e-12 * scale


@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 5, 2), (16, 16, 5), (9, 40, 3), (33, 20, 4),
                                  (41, 25, 5), (32, 32, 5), (64, 32, 5), (33, 63, 5), (64, 64, 3),
                                  (63, 66, 3), (91, 90, 2), (91, 91, 2)])
def test_bond_solves_over_the_vector_lengths(dims):
    """Small bonds in one launch; n = 1024, 1025, 2048, 2079, 4096, 4158, 8190, 8281 through the
    steps on short vectors and beyond them."""
    rng = np.random.default_rng(sum(dims))
    Dl, Dr, M = dims
    l, r = _herm(rng, Dl, M), _herm(rng, Dr, M)
    c = orc.crandn((Dl, Dr), rng)
    k = min(9, c.size)
    hfun = lambda x: orc.apply_local_bond_contraction(x.reshape(c.shape), l, r).reshape(-1)
    got, _, info = _solve(_lib.PTN_OP_BOND, c, l, None, r, k, "expm", 0.07j)
    assert list(info) == [k, 0, 0, 0]
    ref = orc.expm_krylov(hfun, c.reshape(-1), 0.07j, k, hermitian=True).reshape(c.shape)
    assert np.linalg.norm(got - ref) < 1e-11 * np.linalg.norm(ref)
    stack = lambda x: np.stack([x, 2.0 * x, 0.5 * x])
    out, _, _ = backend.krylov_local_batched(_lib.PTN_OP_BOND, stack(c), stack(l), None,
                                             np.stack([r] * 3), k, "expm", 0.07j)
    assert np.linalg.norm(backend.to_host(out)[0] - ref) < 1e-11 * np.linalg.norm(ref)


@pytest.mark.parametrize("dt", [1e-6j, 0.5, -0.5, 3.0j, 1.0 - 2.0j, 40.0j, -6.0 + 20.0j])
def test_exponential_over_the_step_sizes(dt):
    """Few and many Taylor steps and, beyond 16, the eigendecomposition."""
    rng = np.random.default_rng(4)
    l, w, r = _operator(rng, 6, 2, 6, 3, 3)
    l, r = l / np.abs(l).max(), r / np.abs(r).max()
    v = orc.crandn((6, 2, 6), rng)
    hfun = lambda x: orc.apply_local_hamiltonian(x.reshape(v.shape), w, l, r).reshape(-1)
    got, _, _ = _solve(_lib.PTN_OP_HEFF, v, l, w, r, 8, "expm", dt)
    ref = orc.expm_krylov(hfun, v.reshape(-1), dt, 8, hermitian=True).reshape(v.shape)
    assert np.linalg.norm(got - ref) < 1e-11 * np.linalg.norm(ref)


@pytest.mark.parametrize("small", [True, False])
def test_status_words(small):
    """Breakdown in an invariant subspace, zero and non-finite start vectors: as the
    launches per step report them."""
    rng = np.random.default_rng(5)
    l, w, r = _operator(rng, 4, 2, 4, 2, 2)
    kw = {} if small else {"block_sparse": True}
    run = lambda x: _solve(_lib.PTN_OP_HEFF, x, l, w, r, 6, "expm", 0.1j, **kw)
    h = np.zeros((32, 32), dtype=complex)
    for i in range(32):
        e = np.zeros(32, dtype=complex)
        e[i] = 1.0
        h[:, i] = orc.apply_local_hamiltonian(e.reshape(4, 2, 4), w, l, r).reshape(-1)
    lam, u = np.linalg.eigh(h)
    v = (u[:, 3] + 2.0 * u[:, 20]).reshape(4, 2, 4)
    out, _, info = run(v)
    assert list(info) == [2, 2, 0, 0]
    ref = np.exp(0.1j * lam[3]) * u[:, 3] + 2.0 * np.exp(0.1j * lam[20]) * u[:, 20]
    assert np.abs(out.reshape(-1) - ref).max() < 1e-11
    out, _, info = run(np.zeros((4, 2, 4), dtype=complex))
    assert list(info) == [0, 0, 0, 1] and not out.any()
    v[1, 1, 1] = np.nan
    out, _, info = run(v)
    assert list(info) == [0, 0, 1, 0] and not out.any()


def test_large_batches():
    """More problems than two per CU take the launches per step."""
    rng = np.random.default_rng(6)
    l, w, r = _operator(rng, 3, 2, 4, 2, 3)
    v = orc.crandn((600, 3, 2, 4), rng)
    rep = lambda x, n: np.broadcast_to(x, (n,) + x.shape).copy()
    out = {}
    for nb in (200, 600):
        (res, _, _), names = _names(lambda: backend.krylov_local_batched(
            _lib.PTN_OP_HEFF, v[:nb], rep(l, nb), rep(w, nb), rep(r, nb), 5, "expm", 0.2j))
        assert ("k_lz_solve" in names) == (nb == 200)
        out[nb] = backend.to_host(res)
    assert np.abs(out[200] - out[600][:200]).max() < 1e-11 * np.abs(out[200]).max()


def test_mpo_matrices_beyond_the_mix_stay_refused():
    rng = np.random.default_rng(7)
    l, w, r = _operator(rng, 2, 12, 2, 3, 3)
    with pytest.raises(backend.PtnError):
        _solve(_lib.PTN_OP_HEFF, orc.crandn((2, 12, 2), rng), l, w, r, 3, "expm", 0.1j)
