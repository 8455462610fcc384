"""The stream every launch goes to: torch's current stream on the tensor's device, with and
without torch's internal accessor of the raw handle."""

from types import SimpleNamespace

import pytest
import torch

from interattn_amd import ops


def test_public_stream_without_the_accessor(monkeypatch):
    asked = []
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: asked.append(dev) or SimpleNamespace(cuda_stream=1234))
    monkeypatch.setattr(ops, "_raw_stream", None)
    t = torch.zeros(1)
    assert ops._stream(t) == 1234 and asked == [t.device]


def test_accessor_is_asked_for_the_tensors_device(monkeypatch):
    monkeypatch.setattr(ops, "_raw_stream", lambda index: 100 + index)
    assert ops._stream(SimpleNamespace(get_device=lambda: 3)) == 103


@pytest.mark.gpu
@pytest.mark.parametrize("raw", [True, False], ids=["accessor", "public"])
def test_current_stream_of_the_device(raw, device, monkeypatch):
    if not raw:
        monkeypatch.setattr(ops, "_raw_stream", None)
    t = torch.zeros(1, device=device)
    side = torch.cuda.Stream(device)
    assert ops._stream(t) == torch.cuda.current_stream(device).cuda_stream
    with torch.cuda.stream(side):
        assert ops._stream(t) == side.cuda_stream
    assert ops._stream(t) == torch.cuda.current_stream(device).cuda_stream
