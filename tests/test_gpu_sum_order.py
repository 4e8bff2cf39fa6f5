"""
The order of the sums in a complex product (csrc/gemm_impl.h) depends on its shape and
type alone: the same bits with and without tile masks, for operands on and off the
16-byte boundary (loads into LDS or through registers), and with the tile autotuner
on or off, whose candidates all divide k as the rule's choice does.
"""

import re

import numpy as np
import pytest
import torch

import oracle as orc
from pytenet_amd import backend, _lib
from test_gpu_sectors import _operator

pytestmark = pytest.mark.gpu


def _names(fn):
    backend.timing_begin()
    res = fn()
    return res, [x["name"] for x in backend.timing_end()]


@pytest.fixture
def fixed_rule():
    prev = backend.set_autotune(False)
    yield
    backend.set_autotune(prev)


# 1280 and 256 tiles of 64 x 32 in the two products (two and four k groups), ragged too
@pytest.mark.parametrize("Dl,Dr", [(512, 512), (509, 517)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_masked_products_add_in_the_order_of_the_dense_ones(fixed_rule, Dl, Dr, precision):
    rng = np.random.default_rng(Dl)
    a, w, l, r, _ = _operator(rng, Dl, Dr, False)
    dense = backend.to_host(backend.heff_apply(a, w, l, r, precision))
    masked = backend.to_host(backend.heff_apply(a, w, l, r, precision, block_sparse=True))
    assert np.array_equal(masked, dense)


# (M, N, K): two and four groups of k, the last stage of 8 whole, partial or alone in its group
SHAPES = [(701, 701, 64), (701, 701, 71), (701, 701, 257), (701, 701, 263), (701, 701, 321),
          (1280, 1000, 259), (2999, 1500, 67)]


def _off_boundary(x):
    buf = torch.zeros(2 * x.size + 1, dtype=torch.float64, device="cuda")
    buf[1:] = torch.view_as_real(backend.as_dev(x)).reshape(-1)
    return buf


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_sums_do_not_depend_on_the_alignment(fixed_rule, M, N, K):
    rng = np.random.default_rng(M + K)
    A, B = orc.crandn((M, K), rng), orc.crandn((K, N), rng)
    ref, names = _names(lambda: backend.matmul(backend.as_dev(A), backend.as_dev(B)))
    assert any("LdsRing" in n for n in names), names
    out = torch.empty((M, N), dtype=torch.complex128, device="cuda")
    a, b = _off_boundary(A), _off_boundary(B)
    st, names = _names(lambda: _lib.load().ptn_zgemm(
        M, N, K, a.data_ptr() + 8, K, 1, 0, b.data_ptr() + 8, N, 1, 0, backend.ptr(out), N, 1, 0,
        None, 0, backend.stream()))
    assert st == 0 and not any("LdsRing" in n for n in names), names
    assert torch.equal(out, ref)


@pytest.mark.parametrize("M,N,K", SHAPES + [(200, 300, 40), (300, 500, 90)])
def test_tuned_products_divide_k_as_the_rule_does(M, N, K):
    rng = np.random.default_rng(M - K)
    A, B = backend.as_dev(orc.crandn((M, K), rng)), backend.as_dev(orc.crandn((K, N), rng))
    prev = backend.set_autotune(False)
    try:
        ref, rule = _names(lambda: backend.matmul(A, B))
        backend.set_autotune(True)
        tuned, names = _names(lambda: backend.matmul(A, B))
        again = backend.matmul(A, B)
    finally:
        backend.set_autotune(prev)

    def groups(n):   # the k groups of zgemm_kernel<types, tile, groups, layouts>
        return re.search(r", (?:\d+, \d+|WaveTile<\d+>), (?:LdsRing<)?(\d+)", n).group(1)
    assert {groups(n) for n in names} == {groups(n) for n in rule}, (rule, names)
    assert torch.equal(tuned, ref) and torch.equal(again, ref)


def test_tuned_fp32_matvec_has_the_bits_of_the_rule():
    """One group in the first product (1280 tiles, tuned), four in the second."""
    a, w, l, r, _ = _operator(np.random.default_rng(2), 512, 512, False)
    prev = backend.set_autotune(False)
    try:
        ref = backend.heff_apply(a, w, l, r, "fp32")
        backend.set_autotune(True)
        for _ in range(2):
            assert torch.equal(backend.heff_apply(a, w, l, r, "fp32"), ref)
    finally:
        backend.set_autotune(prev)
