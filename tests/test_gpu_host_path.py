"""The device layer's argument handling (pytenet_amd/backend.py): what as_dev returns
for every kind of input, and the current stream as seen by the library."""

import numpy as np
import pytest
import torch

import oracle as orc
from pytenet_amd import backend

pytestmark = pytest.mark.gpu


def test_as_dev_accepts_every_kind_of_input():
    rng = np.random.default_rng(1)
    x = orc.crandn((3, 4, 5), rng)
    t = torch.as_tensor(x, device="cuda")
    assert backend.as_dev(t) is t
    s = t.permute(2, 1, 0)
    for given in (x, x.astype(np.complex64), x.real, x.tolist(), np.asfortranarray(x), s,
                  t.to(torch.complex64), t.cpu(), torch.nn.Parameter(t)):
        got = backend.as_dev(given)
        assert got.dtype == torch.complex128 and got.is_cuda and got.is_contiguous()
        want = np.asarray(given.detach().cpu() if isinstance(given, torch.Tensor) else given)
        assert np.array_equal(backend.to_host(got), want.astype(np.complex128))
    assert complex(backend.as_dev(2.5 - 1j).item()) == 2.5 - 1j


def test_calls_follow_the_current_stream():
    rng = np.random.default_rng(2)
    a, b = orc.crandn((70, 40), rng), orc.crandn((40, 50), rng)
    side = torch.cuda.Stream()
    main = backend.stream()
    with torch.cuda.stream(side):
        assert backend.stream() == side.cuda_stream != main
        got = backend.matmul(backend.as_dev(a), backend.as_dev(b))
    torch.cuda.current_stream().wait_stream(side)
    assert backend.stream() == main
    assert np.abs(backend.to_host(got) - a @ b).max() <= 1e-13 * np.abs(a @ b).max()
