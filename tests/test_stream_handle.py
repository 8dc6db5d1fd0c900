"""The front end's stream handle, on the CPU: torch's raw accessors where it has them, the public call where not."""
import importlib.util
import os
import types

import pytest
import torch

PATH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sam-rs_amd", "sam_hip.py")


def front_end():
    spec = importlib.util.spec_from_file_location("sam_hip_under_test", PATH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("missing", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_public_call_without_the_raw_accessors(monkeypatch, missing):
    monkeypatch.delattr(torch._C, missing, raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=0x1230))
    assert front_end()._stream() == 0x1230


def test_raw_accessors(monkeypatch):
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 3, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda dev: 0x4560 + dev, raising=False)
    assert front_end()._stream() == 0x4563
