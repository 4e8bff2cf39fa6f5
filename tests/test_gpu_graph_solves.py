"""
Captured local solves of more than one launch (ptn_set_graphs, off by default): vectors and
precisions beyond the one-launch solve, a breakdown whose remaining iterations are
predicated off, the reduced-precision products inside a capture, and the buckets of the
batched driver. Every replay, with eager work and synchronisations between them, gives the
bits of the direct launches.
"""

import copy

import numpy as np
import pytest
import torch

import oracle as orc
import pytenet_amd as ptn
from pytenet_amd import backend, _lib
from test_gpu_batched import _herm_env, _herm_w, _padded_chains

pytestmark = pytest.mark.gpu


def _solve(ops, mode, numiter, precision):
    v, l, w, r = ops
    return backend.krylov_local(_lib.PTN_OP_HEFF, v, l, w, r, numiter, mode, -0.05j, precision)


def _captured_equals_direct(problems, mode, numiter, precision):
    """Every problem through one shape bucket, captured and direct; the direct
    launches of a solve must be several."""
    prev = backend.set_graphs(False)
    try:
        backend.timing_begin()
        direct = [_solve(p, mode, numiter, precision) for p in problems]
        launches = sum(x["launches"] for x in backend.timing_end())
        assert launches >= numiter * len(problems)   # (products; k_lz_solve is one for each)
        backend.set_graphs(True)
        n0 = backend.graph_launches()
        got = []
        for p in problems:
            got.append(_solve(p, mode, numiter, precision))
            backend.heff_apply(p[0], p[2], p[1], p[3], precision)
            torch.cuda.synchronize()
        assert backend.graph_launches() - n0 == len(problems)
    finally:
        backend.set_graphs(prev)
    for (o, e, i), (co, ce, ci) in zip(direct, got):
        assert torch.equal(co, o) and torch.equal(ci, i)
        assert e is None or torch.equal(ce, e)
    return [backend.to_host(x[2]) for x in direct]


# 5120 and 20 640 elements (the vector kernels of one workgroup and of many), FP32, and the
# three-term products at the largest vectors that are captured
@pytest.mark.parametrize("Dl,d,Dr,precision,mode,count", [
    (40, 4, 32, "fp64", "expm", 5), (40, 4, 32, "fp64", "eigh", 5), (60, 4, 86, "fp64", "expm", 5),
    (24, 2, 20, "fp32", "expm", 5), (512, 4, 512, "bf16x6", "expm", 4)])
def test_captured_solves_equal_direct_launches(Dl, d, Dr, precision, mode, count):
    problems = []
    for seed in range(count):
        rng = np.random.default_rng(seed)
        a, w = orc.crandn((Dl, d, Dr), rng), _herm_w(rng, 5, d)
        l, r = _herm_env(rng, Dl, 5) / Dl, _herm_env(rng, Dr, 5) / Dr
        problems.append([backend.as_dev(x) for x in (a / np.linalg.norm(a), l, w, r)])
    _captured_equals_direct(problems, mode, 4, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_captured_solve_with_a_breakdown(precision):
    """Start vectors in an invariant subspace of two dimensions: the solve stops after two
    steps, and the captured iterations after it do nothing."""
    D, rng = 40, np.random.default_rng(3)
    one = np.eye(D).reshape(D, 1, D)
    w = np.diag([1.0, 2.0, 3.0, 4.0]).reshape(1, 4, 4, 1)
    problems = []
    for k in range(4):
        a = np.zeros((D, 4, D), dtype=complex)
        a[:, k % 3, :] = orc.crandn((D, D), rng)
        a[:, k % 3 + 1, :] = orc.crandn((D, D), rng)
        problems.append([backend.as_dev(x) for x in (a / np.linalg.norm(a), one, w, one)])
    for info in _captured_equals_direct(problems, "expm", 5, precision):
        assert info[0] == 2 and info[1] == 2 and info[2] == 0


def test_captured_bf16x3_solves_equal_direct_launches():
    """bf16x3 inside a capture (no solve of it takes one launch), bond operator included."""
    rng = np.random.default_rng(9)
    a, w = orc.crandn((512, 2, 512), rng), _herm_w(rng, 5, 2)
    l, r = _herm_env(rng, 512, 5) / 512, _herm_env(rng, 512, 5) / 512
    p = [backend.as_dev(x) for x in (a / np.linalg.norm(a), l, w, r)]
    _captured_equals_direct([p, [0.5 * p[0]] + p[1:]], "expm", 4, "bf16x3")
    c = p[0][:, 0, :].contiguous()
    prev = backend.set_graphs(True)
    try:
        n0 = backend.graph_launches()
        got = [backend.krylov_local(_lib.PTN_OP_BOND, c, p[1], None, p[3], 4, "expm", -0.1j,
                                    "bf16x3")[0] for _ in range(3)]
        assert backend.graph_launches() - n0 == 3
        backend.set_graphs(False)
        ref = backend.krylov_local(_lib.PTN_OP_BOND, c, p[1], None, p[3], 4, "expm", -0.1j,
                                   "bf16x3")[0]
    finally:
        backend.set_graphs(prev)
    assert all(torch.equal(x, ref) for x in got)


def test_batched_buckets_with_captured_solves_equal_direct_launches():
    """The buckets of the batched driver on their streams, FP32 (solves of many launches):
    captured and direct give the same bits."""
    Hs, psis = _padded_chains(6, 10, [4, 8, 16], seed=21)
    direct = [copy.deepcopy(p) for p in psis]
    prev = backend.set_graphs(True)
    try:
        n0 = backend.graph_launches()
        ptn.tdvp_singlesite_batched(Hs, psis, 0.05, 2, numiter_lanczos=6, precision="fp32")
        assert backend.graph_launches() > n0
        backend.set_graphs(False)
        n0 = backend.graph_launches()
        ptn.tdvp_singlesite_batched(Hs, direct, 0.05, 2, numiter_lanczos=6, precision="fp32")
        assert backend.graph_launches() == n0
    finally:
        backend.set_graphs(prev)
    for p, q in zip(psis, direct):
        for x, y in zip(p.a, q.a):
            assert np.array_equal(backend.to_host(x), backend.to_host(y))
