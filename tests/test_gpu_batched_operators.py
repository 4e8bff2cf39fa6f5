"""
The MPO tensors of the batched driver may be host arrays (stacked there, one upload
per site) or tensors, on the device or not, lazily conjugated ones among them.
"""

import copy

import numpy as np
import pytest
import torch

import pytenet_amd as ptn
from pytenet_amd import backend
from test_gpu_batched import _padded_chains

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["device", "conjugated", "host tensors", "mixed"])
def test_operators_as_tensors(kind):
    Hs, psis = _padded_chains(4, 6, [4], seed=5)
    for H in Hs:   # complex entries: a phase on one channel of a bond and its inverse
        H.a = [np.array(t, dtype=np.complex128) for t in H.a]
        H.a[2][..., 1] *= np.exp(0.3j)
        H.a[3][1] *= np.exp(-0.3j)
    got, As = [copy.deepcopy(p) for p in psis], [copy.copy(H) for H in Hs]
    for j, H in enumerate(As):
        if kind == "device" or (kind == "mixed" and j % 2):
            H.a = [torch.as_tensor(t, device="cuda") for t in H.a]
        elif kind == "conjugated":
            H.a = [torch.as_tensor(t.conj(), device="cuda").conj() for t in H.a]
        elif kind == "host tensors":
            H.a = [torch.as_tensor(t.conj()).conj() for t in H.a]
    ptn.tdvp_singlesite_batched(Hs, psis, 0.05, 1, numiter_lanczos=4)
    ptn.tdvp_singlesite_batched(As, got, 0.05, 1, numiter_lanczos=4)
    for p, q in zip(psis, got):
        for x, y in zip(p.a, q.a):
            assert np.array_equal(backend.to_host(x), backend.to_host(y))
