"""
The 128 x 128 tile of the FP32 products (csrc/gemm_impl.h) with every pair of operand types
that the contractions give it: environment steps and H_eff at MPO bond 8 and 16, the
smallest sizes that select it, with a partial last stage, against the oracle.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_batched import _herm_env, _herm_w
from test_gpu_kernels import FP32_TOL, relerr
from test_gpu_tiles_ring import _names

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Dl,Dr,M,types", [
    (512, 509, 16, {"c64, c128, c64", "c128, c64, c64", "c64, c64, c64"}),
    (509, 512, 16, {"c64, c128, c64", "c128, c64, c64", "c64, c64, c64"}),
    (45, 1021, 8, {"c128, c64, c128"}), (1021, 45, 8, {"c64, c128, c128"})])
def test_wide_tiles_match_oracle(Dl, Dr, M, types):
    rng = np.random.default_rng(Dl + M)
    a, b, w = orc.crandn((Dl, 2, Dr), rng), orc.crandn((Dl, 2, Dr), rng), _herm_w(rng, M, 2)
    l, r = _herm_env(rng, Dl, M), _herm_env(rng, Dr, M)
    seen = set()
    for got, ref in (
            (lambda: backend.env_left(a, b, w, l, "fp32"),
             lambda: orc.contraction_operator_step_left(a, b, w, l)),
            (lambda: backend.env_right(a, b, w, r, "fp32"),
             lambda: orc.contraction_operator_step_right(a, b, w, r)),
            (lambda: backend.heff_apply(a, w, l, r, "fp32"),
             lambda: orc.apply_local_hamiltonian(a, w, l, r))):
        x, names = _names(got)
        seen |= {n.split(", 4, 8, 1, ")[0].split("float, ")[1] for n in names if ", 4, 8, 1, " in n}
        assert relerr(x, ref()) < FP32_TOL
    assert seen == types
