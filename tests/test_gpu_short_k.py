"""
FP64 products of a short inner dimension with more tiles than the chip holds at once
(csrc/gemm_impl.h launch_cfg): K from one to the first that loads into LDS again, both tiles, all
layouts, batches and accumulation, against NumPy within the bound of test_gpu_tiles.py.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_tiles import EPS, _dev, _within
from test_gpu_tiles_ring import _names

pytestmark = pytest.mark.gpu


# 64 x 32 tiles: 1278 and, in a batch, 1224; 128 x 64: 1504 (every second K)
@pytest.mark.parametrize("M,N,tile", [(1095, 2249, "2, 2"), (4000, 3000, "4, 4")])
@pytest.mark.parametrize("K", [1, 4, 5, 8, 12, 13, 16, 20, 23, 24])
def test_short_inner_dimensions(M, N, tile, K):
    rng = np.random.default_rng(M + K)
    A, B = orc.crandn((M, K), rng), orc.crandn((K, N), rng)
    ta, tb = bool(K & 1), bool(K & 4)
    prev = backend.set_autotune(False)
    try:
        got, names = _names(lambda: backend.matmul(_dev(A, ta), _dev(B, tb), conjA=tb, conjB=ta))
        out = backend.as_dev(np.full((M, N), 1.0 - 2.0j))
        backend.matmul(_dev(A, tb), _dev(B, ta), out=out, accumulate=True)
    finally:
        backend.set_autotune(prev)
    assert len(names) == 1 and f"{tile}, {1 if K < 24 else 'LdsRing<1>'}," in names[0], names
    _within(backend.to_host(got), A.conj() if tb else A, B.conj() if ta else B, EPS["fp64"])
    _within(backend.to_host(out), A, B, EPS["fp64"], np.full((M, N), 1.0 - 2.0j))


@pytest.mark.parametrize("K", [1, 7, 17])
def test_batches_of_short_inner_dimensions(K):
    rng = np.random.default_rng(K)
    A, B = orc.crandn((18, 250, K), rng), orc.crandn((18, K, 530), rng)
    got, names = _names(lambda: backend.matmul_batched(backend.as_dev(A), backend.as_dev(B)))
    assert len(names) == 1 and "2, 2, 1," in names[0], names
    got = backend.to_host(got)
    for b in range(18):
        _within(got[b], A[b], B[b], EPS["fp64"])
