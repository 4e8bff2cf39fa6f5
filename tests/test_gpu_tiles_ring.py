"""
FP64 products whose stages are loaded straight into LDS (csrc/gemm_impl.h): every
remainder of a stage of 8 k, products shorter than the three stages in flight,
shares of k that leave a group with fewer stages or none, all layouts, operands with
two non-unit strides, and operands off the 16-byte boundary (staged through registers).
Reference and bound: test_gpu_tiles.py.
"""

import numpy as np
import pytest
import torch

import oracle as orc
from pytenet_amd import backend, _lib
from test_gpu_tiles import EPS, _dev, _within

pytestmark = pytest.mark.gpu


def _names(fn):
    backend.timing_begin()
    res = fn()
    return res, [x["name"] for x in backend.timing_end()]


# (M, N), tile; 64 x 32 with 1, 2 and 4 groups by K (and the number of tiles), 128 x 64
CASES = [(701, 701, k, "2, 2, LdsRing<%d>" % (1 if k < 64 else 2 if k < 256 else 4))
         for k in (1, 7, 8, 15, 24, 63, 64, 71, 81, 104, 255, 256, 257, 263, 290, 321)]
CASES += [(1280, 1000, 259, "2, 2, LdsRing<2>"), (2999, 1500, 67, "2, 2, LdsRing<1>")]
CASES += [(4095, 1021, k, "4, 4, LdsRing<1>") for k in (5, 16, 25, 38)]


@pytest.mark.parametrize("M,N,K,tile", CASES)
def test_stage_remainders(M, N, K, tile):
    rng = np.random.default_rng(M + N + K)
    A, B = orc.crandn((M, K), rng), orc.crandn((K, N), rng)
    prev = backend.set_autotune(False)
    try:
        for ta, tb in ((False, False), (True, False), (False, True), (True, True)):
            got, names = _names(lambda: backend.matmul(_dev(A, ta), _dev(B, tb), conjA=tb,
                                                       conjB=ta))
            assert any(tile in n for n in names), names
            _within(backend.to_host(got), A.conj() if tb else A, B.conj() if ta else B, EPS["fp64"])
    finally:
        backend.set_autotune(prev)


@pytest.mark.parametrize("M,N,K", [(700, 650, 50), (700, 650, 301)])
def test_strided_operands_and_accumulation(M, N, K):
    rng = np.random.default_rng(K)
    A, B = orc.crandn((2 * M, 3 * K), rng), orc.crandn((2 * K, 2 * N), rng)
    C = orc.crandn((M, N), rng)
    out = backend.as_dev(C)
    backend.matmul(backend.as_dev(A)[::2, ::3], backend.as_dev(B)[::2, ::2], out=out,
                   accumulate=True)
    _within(backend.to_host(out), A[::2, ::3], B[::2, ::2], EPS["fp64"], C)


def test_operands_off_the_16_byte_boundary():
    rng = np.random.default_rng(1)
    M, N, K = 701, 640, 90
    A, B = orc.crandn((M, K), rng), orc.crandn((K, N), rng)
    dev = []
    for x in (A, B):
        buf = torch.zeros(2 * x.size + 1, dtype=torch.float64, device="cuda")
        buf[1:] = torch.view_as_real(backend.as_dev(x)).reshape(-1)
        dev.append(buf)
    out = torch.empty((M, N), dtype=torch.complex128, device="cuda")
    lib = _lib.load()
    st, names = _names(lambda: lib.ptn_zgemm(
        M, N, K, dev[0].data_ptr() + 8, K, 1, 0, dev[1].data_ptr() + 8, N, 1, 0, backend.ptr(out),
        N, 1, 0, None, 0, backend.stream()))
    assert st == 0 and not any("LdsRing" in n for n in names), names
    _within(backend.to_host(out), A, B, EPS["fp64"])
