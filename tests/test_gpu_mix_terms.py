"""
Mode mix straight into the terms of the three-term split-bf16 product
(csrc/gemm_bf16.hip k_mix_split3): units of 8 x 16 columns with remainders of both,
a last k-block that the product pads, both directions that take it (H_eff, left
environment step) and a batch. Bound: the FP32 bound of these products
(test_gpu_kernels.py); the mixed values and their terms are those of the two passes.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_kernels import FP32_TOL, _heff_problem, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Dl,Dr,d,M", [(521, 529, 4, 5), (603, 607, 4, 5), (520, 512, 4, 4),
                                       (1031, 703, 2, 3)])
def test_mix_into_terms_matches_oracle(Dl, Dr, d, M):
    a, w, l, r = _heff_problem(Dl + Dr + d, Dl=Dl, d=d, Dr=Dr, M=M)
    assert relerr(backend.heff_apply(a, w, l, r, "bf16x6"),
                  orc.apply_local_hamiltonian(a, w, l, r)) < FP32_TOL
    assert relerr(backend.env_left(a, a, w, l, "bf16x6"),
                  orc.contraction_operator_step_left(a, a, w, l)) < FP32_TOL


def test_mix_into_terms_of_a_batch():
    p = [_heff_problem(b, Dl=193, d=2, Dr=193, M=5) for b in range(16)]
    a, w, l = (np.stack([np.asarray(q[i]) for q in p]) for i in range(3))
    got = backend.to_host(backend.env_left_batched(a, w, l, "bf16x6"))
    for b in range(16):
        assert relerr(got[b], orc.contraction_operator_step_left(a[b], a[b], w[b], l[b])) < FP32_TOL
