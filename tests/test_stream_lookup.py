"""The stream and device lookups of a call where torch lacks its private functions (CPU, torch.cuda replaced)."""

import contextlib

import pytest
import torch

from pulsarlm_amd import ops


@pytest.mark.parametrize("current", [0, 1])
def test_lookups_without_private_functions(monkeypatch, current):
    class Stream:
        cuda_stream = 1234

    entered = []

    @contextlib.contextmanager
    def device_guard(device):
        entered.append(device)
        yield

    for name in ("_cuda_getCurrentRawStream", "_cuda_getDevice"):
        monkeypatch.delattr(torch._C, name, raising=False)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: Stream())
    monkeypatch.setattr(torch.cuda, "device", device_guard)
    device = torch.device("cuda", 0)
    assert ops._stream(device) == 1234
    with ops._on(device):
        pass
    assert entered == ([] if current == 0 else [device])
