"""
Environment operands of single three-term split-bf16 calls (csrc/capi.hip
once_operand): the pre-split product reads them in complex128, the other products
after a conversion to complex64. Both round every value to FP32 first, so operands
that are rounded beforehand give the same bits, on each route; and the results stay
within the FP32 bound of these products (test_gpu_kernels.py) of the oracle.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend
from test_gpu_kernels import FP32_TOL, _heff_problem, relerr

pytestmark = pytest.mark.gpu


def _fp32(x):
    return np.asarray(x).astype(np.complex64).astype(np.complex128)


# H_eff: neither product pre-split, the first, both
@pytest.mark.parametrize("Dl,Dr", [(40, 36), (384, 385), (601, 600)])
def test_single_calls_round_their_operands_to_fp32(Dl, Dr):
    a, w, l, r = _heff_problem(Dl + 3 * Dr, Dl=Dl, d=4, Dr=Dr, M=5)
    l, r = np.asarray(l), np.asarray(r)
    c = orc.crandn((Dl, Dr), np.random.default_rng(Dl))
    calls = [
        (lambda l, r: backend.heff_apply(a, w, l, r, "bf16x6"),
         orc.apply_local_hamiltonian(a, w, l, r)),
        (lambda l, r: backend.env_left(a, a, w, l, "bf16x6"),
         orc.contraction_operator_step_left(a, a, w, l)),
        (lambda l, r: backend.env_right(a, a, w, r, "bf16x6"),
         orc.contraction_operator_step_right(a, a, w, r)),
        (lambda l, r: backend.bond_apply(c, l, r, "bf16x6"),
         orc.apply_local_bond_contraction(c, l, r)),
    ]
    for call, ref in calls:
        got = backend.to_host(call(l, r))
        assert np.array_equal(got, backend.to_host(call(_fp32(l), _fp32(r))))
        assert relerr(got, ref) < FP32_TOL


@pytest.mark.parametrize("D", [33, 193])
def test_batched_steps_round_their_operands_to_fp32(D):
    p = [_heff_problem(D + b, Dl=D, d=2, Dr=D, M=5) for b in range(12)]
    a, w, l, r = (np.stack([np.asarray(q[i]) for q in p]) for i in range(4))
    for step, e in ((backend.env_left_batched, l), (backend.env_right_batched, r)):
        got = backend.to_host(step(a, w, e, "bf16x6"))
        assert np.array_equal(got, backend.to_host(step(a, w, _fp32(e), "bf16x6")))
