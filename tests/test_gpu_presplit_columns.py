"""
Three-term split-bf16 products whose B operand is held once per complex column and
embedded from the fragments (csrc/gemm_bf16.hip): one column more and one fewer than
the 128 of a tile, one k-stage more or fewer in the last chunk of k, conjugated and
strided operands (both environment steps). Bound: the FP32 bound of these products
(test_gpu_kernels.py); the embedding only moves and negates terms.
"""

import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_kernels import FP32_TOL, _heff_problem, relerr

pytestmark = pytest.mark.gpu


# columns 5 Dr: 13 * 128 + 1, 17 * 128 - 1, 15 * 128 (full tiles)
@pytest.mark.parametrize("Dl,Dr", [(333, 333), (261, 435), (384, 384)])
def test_embedded_columns_at_tile_edges(Dl, Dr):
    a, w, l, r = _heff_problem(Dl + 2 * Dr, Dl=Dl, d=4, Dr=Dr, M=5)
    backend.timing_begin()
    got = [backend.heff_apply(a, w, l, r, "bf16x6"), backend.env_left(a, a, w, l, "bf16x6"),
           backend.env_right(a, a, w, r, "bf16x6")]
    names = [t["name"] for t in backend.timing_end()]
    # the first product of each (the second has too few tiles for this kernel)
    assert "zgemm_bf16x6_v3<c64>" in names, names
    ref = [orc.apply_local_hamiltonian(a, w, l, r),
           orc.contraction_operator_step_left(a, a, w, l),
           orc.contraction_operator_step_right(a, a, w, r)]
    for g, x in zip(got, ref):
        assert relerr(g, x) < FP32_TOL
