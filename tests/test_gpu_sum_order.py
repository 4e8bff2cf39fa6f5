"""
The order of the sums in a complex product (csrc/gemm_impl.h) depends on its shape and
type alone: the same bits with and without tile masks.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_sectors import _operator

pytestmark = pytest.mark.gpu


@pytest.fixture
def fixed_rule():
    prev = backend.set_autotune(False)
    yield
    backend.set_autotune(prev)


# 1280 and 256 tiles of 64 x 32 in the two products (two and four k groups)
@pytest.mark.parametrize("Dl,Dr", [(512, 512)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_masked_products_add_in_the_order_of_the_dense_ones(fixed_rule, Dl, Dr, precision):
    rng = np.random.default_rng(Dl)
    a, w, l, r, _ = _operator(rng, Dl, Dr, False)
    dense = backend.to_host(backend.heff_apply(a, w, l, r, precision))
    masked = backend.to_host(backend.heff_apply(a, w, l, r, precision, block_sparse=True))
    assert np.array_equal(masked, dense)
