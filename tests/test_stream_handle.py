"""The stream handle that the operators launch on."""
import types

import pytest
import torch

from ccinfer_amd import ops


@pytest.mark.parametrize("missing", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_without_the_private_calls(monkeypatch, missing):
    """torch's calls below current_stream() are not public: without them its handle is used."""
    monkeypatch.delattr(torch._C, missing, raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda: types.SimpleNamespace(cuda_stream=1234))
    assert ops._stream_reader()() == 1234


@pytest.mark.gpu
def test_follows_the_current_stream(gpu):
    side = torch.cuda.Stream()
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert ops._stream() == side.cuda_stream
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
