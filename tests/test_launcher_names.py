"""The run calls find the current stream where torch lacks the names that are not public."""
import torch

import cutespmm_ae_amd as cs


class _Stream:
    def __init__(self, handle):
        self.cuda_stream = handle


def _handles(monkeypatch, keep):
    for name, value in (("_cuda_getDevice", lambda: 3), ("_cuda_getCurrentRawStream", lambda d: 1000 + d)):
        if keep:
            monkeypatch.setattr(torch._C, name, value, raising=False)
        else:
            monkeypatch.delattr(torch._C, name, raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: _Stream(1000 + d))
    cs._launcher.cache_clear()
    try:
        _, _, stream_handle = cs._launcher()
        return stream_handle(None), stream_handle(_Stream(7))
    finally:
        cs._launcher.cache_clear()


def test_current_stream_with_and_without_the_private_names(monkeypatch):
    assert _handles(monkeypatch, True) == (1003, 7)
    assert _handles(monkeypatch, False) == (1003, 7)
