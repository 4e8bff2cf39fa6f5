"""
The groups of k of batched FP64 products (csrc/gemm_impl.h k_groups): one group from 256 tiles
of 64 x 32 in a batch on up to K = 1024, two or four on either side of that; at
each edge against NumPy, within the bound of test_gpu_tiles.py.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_tiles import EPS, _within
from test_gpu_tiles_ring import _names

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,M,N,K,groups", [
    (8, 128, 512, 65, 1), (17, 65, 255, 130, 1), (5, 128, 800, 130, 2), (2, 512, 500, 1024, 1),
    (2, 509, 512, 1025, 4), (2, 449, 509, 300, 1), (3, 190, 1000, 257, 1), (3, 190, 900, 257, 1),
    (3, 190, 800, 257, 4)])
def test_groups_of_batched_products(nb, M, N, K, groups):
    rng = np.random.default_rng(nb + M + K)
    A, B = orc.crandn((nb, M, K), rng), orc.crandn((nb, K, N), rng)
    prev = backend.set_autotune(False)
    try:
        got, names = _names(lambda: backend.matmul_batched(backend.as_dev(A), backend.as_dev(B)))
    finally:
        backend.set_autotune(prev)
    assert len(names) == 1 and "2, 2, LdsRing<%d>" % groups in names[0], names
    got = backend.to_host(got)
    for b in range(nb):
        _within(got[b], A[b], B[b], EPS["fp64"])
