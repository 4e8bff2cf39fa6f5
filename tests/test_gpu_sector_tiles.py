"""
The tiles, the zero fill and the mix of the sector-grouped products where they can go
wrong: sector sizes at the edges of the 16 / 32 / 64 / 128 tiles and of the
k stages, units of the mix with more rows and columns than one workgroup takes,
and an output in the memory of an input. FP64: 1e-12 of the largest entry
(sums of < 2^13 products of entries of order one, 2^-53 sqrt(2^13) ~ 1e-14 of
it, with the summation order free), FP32: 2e-5 (2^-24 sqrt(2^13) = 5e-6).
"""

import ctypes

import numpy as np
import pytest

import oracle as orc
from pytenet_amd import backend, _lib
from test_gpu_sectors import TOL, _operator, _qsparse, relerr

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 33, 63, 65, 127, 129, 64, 32]


def _labels(sizes, parity=0):
    return 2 * np.repeat(np.arange(len(sizes)) - len(sizes) // 2, sizes) + parity


def _case(sizes, two_site, seed):
    rng = np.random.default_rng(seed)
    ql, qr = _labels(sizes), _labels(sizes[::-1], 0 if two_site else 1)
    return rng, _operator(rng, len(ql), len(qr), two_site, ql=ql, qr=qr)


@pytest.mark.parametrize("sizes,two_site,tile", [
    ([1, 2, 1], True, 1), ([15, 17, 16], False, 1), (EDGES, False, None), (EDGES, True, None),
    ([70, 100, 130, 160, 130, 100, 70], True, None),
    ([127, 128, 126, 128, 125, 128, 128, 124], True, 2)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_sector_edges(sizes, two_site, tile, precision):
    rng, (a, w, l, r, q) = _case(sizes, two_site, sum(sizes))
    backend.timing_begin()
    out, grouped = backend.heff_apply_sectors(a, w, l, r, q, precision)
    names = [x["name"] for x in backend.timing_end() if x["name"].startswith("zgemm_grouped")]
    assert grouped
    if tile is not None:
        assert any(", %d, %d, " % (tile, tile) in n for n in names), names
    assert relerr(out, orc.apply_local_hamiltonian(a, w, l, r)) < TOL[precision]
    off = np.add.outer(np.add.outer(q[0], q[1]), -q[2]) != 0
    assert np.all(backend.to_host(out)[off] == 0)
    b = _qsparse(rng, a.shape, [q[0], q[1], -q[2]])
    for side, blk, ref in (
            (_lib.PTN_ENV_LEFT, l, orc.contraction_operator_step_left(a, b, w, l)),
            (_lib.PTN_ENV_RIGHT, r, orc.contraction_operator_step_right(a, b, w, r))):
        got, grouped = backend._env_sectors(side, backend.as_dev(a), backend.as_dev(b),
                                            backend.as_dev(w), backend.as_dev(blk), q, precision,
                                            ref.shape)
        assert grouped
        assert relerr(got, ref) < TOL[precision]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_output_in_place_of_the_tensor(precision):
    """ptn_local_apply with out = the tensor it is applied to (FP64 and FP32):
    the zero fill must not run before the first product has read it."""
    _, (a, w, l, r, q) = _case([15, 33, 64, 20], True, 3)
    ref = orc.apply_local_hamiltonian(a, w, l, r)
    a, w, l, r = (backend.as_dev(x).clone() for x in (a, w, l, r))
    Dl, d, Dr = a.shape
    op, keep = backend._local_op(_lib.PTN_OP_HEFF, precision, l, w, r, Dl, d, Dr, True, q)
    lib = _lib.load()
    ws = backend.workspace(lib.ptn_heff_workspace(op.precision, Dl, d, Dr, w.shape[0], w.shape[3]))
    grouped = ctypes.c_int32(0)
    assert lib.ptn_local_apply(ctypes.byref(op), backend.ptr(a), backend.ptr(a),
                               ctypes.addressof(grouped), backend.ptr(ws), ws.numel(),
                               backend.stream()) == 0
    assert grouped.value
    assert relerr(a, ref) < TOL[precision]
    del keep
