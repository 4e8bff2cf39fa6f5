"""
The tile shapes and k-splits of the complex products (csrc/gemm_impl.h), each at
sizes where it can go wrong: one past and one short of its tile edges, partial
k-stages, shares of k that leave a group or wave without work, every layout of
the operands, batches, accumulation and the largest product of its range.
Reference: NumPy in complex128; every output is held to the bound of a sum of
n = 4 K rounded products, n eps (|A| |B|), with a factor of two to spare.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend

pytestmark = pytest.mark.gpu

EPS = {"fp64": np.finfo(np.float64).eps, "fp32": np.finfo(np.float32).eps}


def _dev(x, trans):
    """Device matrix equal to x, stored row-major or as the transpose of one."""
    if trans:
        return backend.as_dev(np.ascontiguousarray(x.T)).transpose(0, 1)
    return backend.as_dev(x)


def _within(got, A, B, eps, C=None):
    ref = A @ B
    bound = 8 * A.shape[-1] * eps * (np.abs(A) @ np.abs(B))
    if C is not None:
        ref, bound = ref + C, bound + 2 * eps * np.abs(C)
    assert np.all(np.abs(got - ref) <= bound)


# (M, N, K) and the tile that the rule takes
SHAPES = [(1, 1, 1), (16, 8, 4), (17, 9, 5), (31, 65, 191), (64, 256, 193), (255, 160, 321),  # wave
          (33, 1000, 37), (513, 497, 63), (160, 401, 65), (129, 321, 255), (161, 335, 257),  # 32 x 16
          (130, 300, 1030),
          (1217, 1025, 40), (450, 900, 100), (449, 993, 513), (700, 1030, 2049),             # 64 x 32
          (1281, 1000, 81),
          (2048, 2040, 73)]                                                                   # 128 x 64


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_products_at_tile_edges(M, N, K, ta, tb):
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    A, B = orc.crandn((M, K), rng), orc.crandn((K, N), rng)
    prev = backend.set_autotune(False)
    try:
        got = backend.to_host(backend.matmul(_dev(A, ta), _dev(B, tb), conjA=ta, conjB=tb))
        C = orc.crandn((M, N), rng)
        out = backend.as_dev(C)
        backend.matmul(_dev(A, ta), _dev(B, tb), out=out, accumulate=True)
    finally:
        backend.set_autotune(prev)
    _within(got, A.conj() if ta else A, B.conj() if tb else B, EPS["fp64"])
    _within(backend.to_host(out), A, B, EPS["fp64"], C)


@pytest.mark.parametrize("nb,M,N,K", [(3, 17, 9, 5), (8, 64, 96, 32), (24, 64, 48, 257),
                                      (70, 33, 47, 12)])
def test_batched_products_at_tile_edges(nb, M, N, K):
    rng = np.random.default_rng(nb + M)
    A, B = orc.crandn((nb, M, K), rng), orc.crandn((nb, K, N), rng)
    got = backend.to_host(backend.matmul_batched(backend.as_dev(A), backend.as_dev(B)))
    for b in range(nb):
        _within(got[b], A[b], B[b], EPS["fp64"])


def test_columns_beyond_the_matrix_do_not_leak():
    """Edge tiles read the last row and column again: non-finite entries there must
    stay in their own row and column."""
    rng = np.random.default_rng(5)
    for M, N, K in ((17, 9, 6), (161, 335, 257), (450, 900, 100)):
        A, B = orc.crandn((M, K), rng), orc.crandn((K, N), rng)
        A[-1, 0], B[1, -1] = np.inf, np.nan
        got = backend.to_host(backend.matmul(backend.as_dev(A), backend.as_dev(B)))
        _within(got[:-1, :-1], A[:-1], B[:, :-1], EPS["fp64"])
        assert not np.isfinite(got[-1]).any() and not np.isfinite(got[:, -1]).any()


@pytest.mark.parametrize("Dl,Dr", [(9, 7), (40, 33), (70, 130), (129, 97), (260, 240), (301, 517)])
@pytest.mark.parametrize("d", [2, 4])
def test_fp32_contractions_over_the_tile_rules(Dl, Dr, d):
    """FP32 H_eff at bond sizes whose products pass through every FP32 tile below
    the largest; relative 2e-5 as for the other FP32 contractions."""
    rng = np.random.default_rng(Dl + Dr)
    a, w = orc.crandn((Dl, d, Dr), rng), orc.crandn((5, d, d, 5), rng)
    l, r = orc.crandn((Dl, 5, Dl), rng), orc.crandn((Dr, 5, Dr), rng)
    ref = orc.apply_local_hamiltonian(a, w, l, r)
    got = backend.to_host(backend.heff_apply(a, w, l, r, "fp32"))
    assert np.abs(got - ref).max() <= 2e-5 * np.abs(ref).max()


@pytest.mark.parametrize("Dl,Dr,d,Ml,Mr", [(1, 1, 2, 1, 1), (3, 15, 2, 5, 5), (7, 16, 2, 3, 5),
                                           (5, 17, 2, 5, 4), (4, 32, 4, 5, 5), (3, 33, 4, 8, 8),
                                           (9, 64, 4, 4, 8), (2, 65, 3, 5, 10), (301, 517, 2, 5, 5)])
def test_mode_mix_units(Dl, Dr, d, Ml, Mr):
    """The mode mix at the edges of its column units (16, 32 and 64 columns, several
    rows per unit, more units than workgroups), with the largest and smallest index
    pairs, and read transposed (left environment); W mostly zero, as an MPO's."""
    rng = np.random.default_rng(Dl * 1000 + Dr)
    a, b = orc.crandn((Dl, d, Dr), rng), orc.crandn((Dl, d, Dr), rng)
    w = orc.crandn((Ml, d, d, Mr), rng) * (rng.random((Ml, d, d, Mr)) < 0.2)
    l, r = orc.crandn((Dl, Ml, Dl), rng), orc.crandn((Dr, Mr, Dr), rng)
    for got, ref in ((backend.heff_apply(a, w, l, r), orc.apply_local_hamiltonian(a, w, l, r)),
                     (backend.env_left(a, b, w, l), orc.contraction_operator_step_left(a, b, w, l)),
                     (backend.env_right(a, b, w, r),
                      orc.contraction_operator_step_right(a, b, w, r))):
        assert np.abs(backend.to_host(got) - ref).max() <= 1e-12 * max(np.abs(ref).max(), 1e-300)
