"""The stream hand-off of the Python calls, with and without torch's raw-handle call."""
import types

import pytest
import torch

from praghip import _util


@pytest.mark.parametrize("raw", [True, False])
def test_current_stream_handle(monkeypatch, raw):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=70))
    if raw:
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 67 + device, raising=False)
    else:
        monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    _util._current_handle.cache_clear()
    try:
        assert _util.stream_handle(None) == 70
        assert _util.stream_handle(types.SimpleNamespace(cuda_stream=5)) == 5
        assert _util.stream_handle(types.SimpleNamespace(cuda_stream=0)) is None  # the null stream
    finally:
        _util._current_handle.cache_clear()
