"""Host side of the Python API that needs no GPU."""
import importlib.util
import types

import torch

from gputils_amd import api


def test_stream_handle_without_the_private_call(monkeypatch):
    """A torch without the raw-stream call: the public stream object's handle."""
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    spec = importlib.util.spec_from_file_location("gputils_amd.api_copy", api.__file__)
    copy = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(copy)
    assert copy.stream_handle() == 77
