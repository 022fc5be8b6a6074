"""The launch stream's raw handle with and without torch's private accessor (CPU)."""
from __future__ import annotations

import importlib.util
from types import SimpleNamespace

import pytest
import torch

from k8v4_v030 import ops_api


@pytest.mark.parametrize("private", [True, False])
def test_the_public_call_serves_where_the_private_one_is_missing(monkeypatch, private):
    if private:
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 100 + index, raising=False)
    else:
        monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: SimpleNamespace(cuda_stream=200 + dev.index))
    spec = importlib.util.find_spec(ops_api.__name__)
    fresh = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(fresh)
    assert fresh._stream(torch.device("cuda", 3)) == (103 if private else 203)
