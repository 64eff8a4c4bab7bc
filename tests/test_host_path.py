"""The per-call host path: the default block is the library's for every domain,
and a call without a stream runs on torch's current one."""
from __future__ import annotations

import types

import pytest
import torch

import lbcube


@pytest.mark.parametrize("lattice", sorted(lbcube.LATTICES))
@pytest.mark.parametrize("extents", [(1, 1, 1), (64, 64, 1), (253, 191, 167), (4096, 2048, 1)])
def test_default_block_is_the_library_s(lattice, extents):
    assert lbcube.default_block(lattice, *extents) == lbcube.DEFAULT_BLOCK
    assert lbcube._block(lattice, None, *extents) == lbcube.DEFAULT_BLOCK
    assert lbcube._block(lattice, [64, 2, 1], *extents) == (64, 2, 1)


@pytest.mark.gpu
def test_current_stream_is_torch_s(gpu):
    assert lbcube._stream(None) == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert lbcube._stream(None) == side.cuda_stream == lbcube._stream(side)
    assert lbcube._stream(None) == torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("name", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_current_stream_without_torchs_private_names(monkeypatch, name):
    monkeypatch.delattr(torch._C, name, raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    assert lbcube._stream(None) == 77
