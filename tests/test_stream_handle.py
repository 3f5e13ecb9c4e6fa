"""The stream that an operator call goes to (xllms_amd.paged_attention): a
given stream or handle, else torch's current stream, whose raw handle comes
from two torch calls that are not public and may be missing."""
from __future__ import annotations

import types

import pytest

from xllms_amd import paged_attention as PA

torch = pytest.importorskip("torch")


@pytest.fixture
def current(monkeypatch):
    """An initialised device 1 whose current stream has handle 71."""
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=71))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 1, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: 70 + d, raising=False)
    return monkeypatch


def test_given_streams(current):
    assert PA._stream_handle(5) == 5
    assert PA._stream_handle(types.SimpleNamespace(cuda_stream=9)) == 9


def test_current_stream(current):
    assert PA._stream_handle(None) == 71


@pytest.mark.parametrize("name", ["_cuda_getDevice", "_cuda_getCurrentRawStream"])
def test_current_stream_without_the_raw_calls(current, name):
    current.delattr(torch._C, name)
    assert PA._stream_handle(None) == 71
