"""Which stream a call without one takes (s14._stream): torch's current
stream, the null stream without torch or a GPU, and torch's own error where
its GPU state cannot be initialised, on every call.  torch is a stand-in."""

from __future__ import annotations

import sys
import types

import pytest

from colormlm_amd import s14


@pytest.fixture
def fake_torch(monkeypatch):
    def install(available=True, init_error=None, raw=True):
        def init():
            if init_error is not None:
                raise init_error

        def device():
            init()
            return 3

        def current_stream():
            init()
            return types.SimpleNamespace(cuda_stream=0x1003)

        cuda = types.SimpleNamespace(is_available=lambda: available, init=init, current_stream=current_stream)
        c = types.SimpleNamespace()
        if raw:
            c._cuda_getDevice, c._cuda_getCurrentRawStream = device, lambda d: 0x1000 + d
        monkeypatch.setitem(sys.modules, "torch", types.SimpleNamespace(cuda=cuda, _C=c))

    monkeypatch.setattr(s14, "_CURRENT_STREAM", [])
    return install


@pytest.mark.parametrize("raw", [True, False])
def test_the_current_stream(fake_torch, raw):
    fake_torch(raw=raw)
    assert s14._stream(None) == 0x1003 and s14._stream(None) == 0x1003
    assert s14._stream(7) == 7 and s14._stream(0) == 0


def test_no_gpu_and_no_torch_take_the_null_stream(fake_torch, monkeypatch):
    fake_torch(available=False)
    assert s14._stream(None) is None
    monkeypatch.setitem(sys.modules, "torch", None)  # import torch raises
    monkeypatch.setattr(s14, "_CURRENT_STREAM", [])
    assert s14._stream(None) is None


@pytest.mark.parametrize("raw", [True, False])
def test_a_failed_initialisation_is_raised_every_time(fake_torch, raw):
    fake_torch(init_error=RuntimeError("HIP initialisation failed"), raw=raw)
    for _ in range(2):
        with pytest.raises(RuntimeError, match="HIP initialisation failed"):
            s14._stream(None)
