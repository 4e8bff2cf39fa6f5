"""
The zero fill of the output inside the first grouped product's launch: groups of 32
fill workgroups (16384 entries each) among the groups of 32 tiles, at sizes whose last
groups are partial on both sides, into an output that holds NaN before the call.
FP64: 1e-12 of the largest entry (sums of < 2^13 products of entries of order one,
2^-53 sqrt(2^13) ~ 1e-14 of it).

The placement: with three sectors at D = 2048 the environment step's fill is 1280
workgroups among 1452 tiles, H_eff's 512 among the same tiles of the same product. Neither
takes more than about 55 us by itself beside a product of about 1.2 ms, so the two launches
may differ by 5 %; spread one by one the environment's took 1.57 times as long. Limit 1.25.
"""

import ctypes

import numpy as np
import pytest
import torch

import oracle as orc
from pytenet_amd import backend, _lib
from test_gpu_sectors import _operator, _qsparse, relerr

pytestmark = pytest.mark.gpu


def _labels(D, ns, parity=0):
    return 2 * (np.arange(D) * ns // D) - ns + parity


# entries of the outputs / 16384: below one workgroup, 1 .. 33 and some more, with few and
# with many tiles
@pytest.mark.parametrize("D,ns", [(8, 2), (57, 3), (58, 3), (129, 40), (325, 3), (331, 25)])
@pytest.mark.parametrize("side", [_lib.PTN_ENV_LEFT, _lib.PTN_ENV_RIGHT])
def test_fill_edges(D, ns, side):
    rng = np.random.default_rng(D)
    ql, qr = _labels(D, ns), _labels(D, ns, 1)
    a, w, l, r, q = _operator(rng, D, D, False, ql=ql, qr=qr)
    b = _qsparse(rng, a.shape, [q[0], q[1], -q[2]])
    left = side == _lib.PTN_ENV_LEFT
    ref = orc.contraction_operator_step_left(a, b, w, l) if left else \
        orc.contraction_operator_step_right(a, b, w, r)
    a, b, w, l, r = (backend.as_dev(x) for x in (a, b, w, l, r))
    op, keep = backend._local_op(_lib.PTN_OP_HEFF, "fp64", l if left else None, w,
                                 None if left else r, D, a.shape[1], D, True, q)
    lib = _lib.load()
    n = ref.size
    out = torch.full((n + 64,), float("nan"), dtype=torch.complex128, device=backend.device())
    ws = backend.workspace(lib.ptn_env_workspace(op.precision, D, a.shape[1], D, op.Ml, op.Mr))
    grouped = ctypes.c_int32(0)
    backend._check(lib.ptn_env_apply(ctypes.byref(op), side, backend.ptr(a), backend.ptr(b),
                                     backend.ptr(out), ctypes.addressof(grouped), backend.ptr(ws),
                                     ws.numel(), backend.stream()), "ptn_env_apply")
    del keep
    assert grouped.value
    got = backend.to_host(out)
    assert np.all(np.isnan(got[n:]))
    got = got[:n].reshape(ref.shape)
    assert relerr(got, ref) < 1e-12
    qm, qo = (q[4], q[2]) if left else (q[3], q[0])
    off = np.add.outer(np.add.outer(qo, qm), -qo) != 0
    assert np.all(got[off] == 0)


def test_fill_leaves_the_product_alone():
    D, ns = 2048, 3
    rng = np.random.default_rng(1)
    ql, qr = _labels(D, ns), _labels(D, ns, 1)
    qs, qm = np.array([1, -1]), np.array([0, 2, -2, 0, 0])
    q = (ql, qs, qr, qm, qm)
    w = backend.as_dev(_qsparse(rng, (5, 2, 2, 5), [qm, qs, -qs, -qm]))
    g = torch.Generator(device=backend.device()).manual_seed(1)

    def dev(*shape):
        return torch.randn(shape, dtype=torch.complex128, device=backend.device(), generator=g)

    a, l, r = dev(D, 2, D), dev(D, 5, D), dev(D, 5, D)
    calls = {"heff": lambda: backend.heff_apply_sectors(a, w, l, r, q, "fp64")[1],
             "env": lambda: backend._env_sectors(_lib.PTN_ENV_RIGHT, a, a, w, r, q, "fp64",
                                                 (D, 5, D))[1]}
    best = {}
    for _ in range(3):
        for what, call in calls.items():
            assert call()
            backend.timing_begin()
            call()
            first = [x for x in backend.timing_end() if x["name"].endswith("4, 4, true, true>")]
            assert len(first) == 1 and first[0]["launches"] == 1
            best[what] = min(best.get(what, 1e9), first[0]["total_ms"])
    assert best["env"] < 1.25 * best["heff"], best
