"""
H_eff and the environment steps of small bonds in one launch (csrc/fused.hip): bonds that
the ranges of a workgroup do not divide, single columns and rows, MPO tensors with empty
rows and single entries, asymmetric bonds, an output in the memory of an input (three
launches then), and the H_eff step through a batch. Against the oracle's contractions; sums of
fewer than 2^11 products, 1e-13 of the largest entry.
"""

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend, _lib

pytestmark = pytest.mark.gpu


def _names(fn):
    backend.timing_begin()
    res = fn()
    return backend.to_host(res), [x["name"] for x in backend.timing_end()]


def _operands(rng, Dl, Dr, d, Ml, Mr):
    w = orc.crandn((Ml, d, d, Mr), rng)
    w *= (rng.uniform(size=(Ml, d, 1, Mr)) < 0.4)      # empty rows and columns
    w[0, 0, 0, 0] = 1.0 + 0.5j
    a, b = orc.crandn((Dl, d, Dr), rng), orc.crandn((Dl, d, Dr), rng)
    return a, b, w, orc.crandn((Dl, Ml, Dl), rng), orc.crandn((Dr, Mr, Dr), rng)


DIMS = [(1, 1, 1, 1, 1), (1, 7, 2, 3, 5), (9, 1, 2, 5, 3), (3, 5, 2, 1, 1), (8, 13, 4, 5, 5),
        (17, 15, 2, 3, 4), (24, 24, 2, 5, 5), (13, 31, 2, 5, 3), (31, 9, 2, 3, 5), (16, 16, 8, 4, 4),
        (5, 6, 16, 2, 2), (6, 40, 2, 3, 3)]


@pytest.mark.parametrize("dims", DIMS)
def test_contractions_of_small_bonds(dims):
    rng = np.random.default_rng(sum(dims) * 3)
    Dl, Dr, d, Ml, Mr = dims
    a, b, w, l, r = _operands(rng, *dims)
    for got, ref, kind in (
            (_names(lambda: backend.heff_apply(a, w, l, r)),
             orc.apply_local_hamiltonian(a, w, l, r), "heff"),
            (_names(lambda: backend.env_left(a, b, w, l)),
             orc.contraction_operator_step_left(a, b, w, l), "left"),
            (_names(lambda: backend.env_right(a, b, w, r)),
             orc.contraction_operator_step_right(a, b, w, r), "right")):
        out, names = got
        if max(Dl, Dr) <= 24 and d <= 4:
            assert names == ["k_fused_apply<%s>" % kind], (kind, names)
        assert np.abs(out - ref).max() <= 1e-13 * max(np.abs(ref).max(), 1e-300)


def test_larger_bonds_take_three_launches():
    rng = np.random.default_rng(2)
    a, b, w, l, r = _operands(rng, 64, 64, 2, 5, 5)
    out, names = _names(lambda: backend.env_left(a, b, w, l))
    assert not any("k_fused_apply" in n for n in names)
    ref = orc.contraction_operator_step_left(a, b, w, l)
    assert np.abs(out - ref).max() <= 1e-13 * np.abs(ref).max()


def test_output_over_an_input():
    """ptn_heff_apply with out = the tensor it is applied to: as before, in place."""
    rng = np.random.default_rng(3)
    a, _, w, l, r = _operands(rng, 12, 10, 2, 3, 4)
    ref = orc.apply_local_hamiltonian(a, w, l, r)
    a, w, l, r = (backend.as_dev(x).clone() for x in (a, w, l, r))
    lib = _lib.load()
    ws = backend.workspace(lib.ptn_heff_workspace(0, 12, 2, 10, 3, 4))
    assert lib.ptn_heff_apply(0, 12, 2, 10, 3, 4, backend.ptr(l), backend.ptr(w), backend.ptr(r),
                              backend.ptr(a), backend.ptr(a), backend.ptr(ws), ws.numel(),
                              backend.stream()) == 0
    assert np.abs(backend.to_host(a) - ref).max() <= 1e-13 * np.abs(ref).max()


def test_batched_steps():
    rng = np.random.default_rng(4)
    ops = [_operands(rng, 11, 14, 2, 3, 5) for _ in range(3)]
    a, _, w, l, r = (backend.as_dev(np.stack([o[k] for o in ops])) for k in range(5))
    left, right = backend.env_left_batched(a, w, l), backend.env_right_batched(a, w, r)
    for k, o in enumerate(ops):
        ref = orc.contraction_operator_step_left(o[0], o[0], o[2], o[3])
        assert np.abs(backend.to_host(left)[k] - ref).max() <= 1e-13 * np.abs(ref).max()
        ref = orc.contraction_operator_step_right(o[0], o[0], o[2], o[4])
        assert np.abs(backend.to_host(right)[k] - ref).max() <= 1e-13 * np.abs(ref).max()
