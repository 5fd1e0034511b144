"""Where HipBackend._stream takes its handle from, without a GPU."""
import sys
from types import SimpleNamespace

import pytest

from oxinfer_amd import HipBackend, hip


def test_torch_is_asked_to_initialise_the_device(monkeypatch):
    """Torch's lazy initialisation, which also refuses a child forked after it, comes before the handle."""
    import torch

    def refuse():
        raise RuntimeError("initialisation was asked for")
    monkeypatch.setattr(hip, "_torch", torch)
    monkeypatch.setattr(torch.cuda, "_lazy_init", refuse)
    if torch.cuda.is_initialized():
        pytest.skip("the device is in use by this process")
    with pytest.raises(RuntimeError, match="asked for"):
        HipBackend._stream()


@pytest.mark.parametrize("accessor,handle", [(True, 11), (False, 22)])
def test_the_handle_without_torchs_accessor(monkeypatch, accessor, handle):
    c = SimpleNamespace(_cuda_getDevice=lambda: 3)
    if accessor:
        c._cuda_getCurrentRawStream = lambda device: {3: 11}[device]
    cuda = SimpleNamespace(current_stream=lambda: SimpleNamespace(cuda_stream=22))
    monkeypatch.setattr(hip, "_torch", SimpleNamespace(_C=c, cuda=cuda))
    assert HipBackend._stream() == handle


def test_without_torch_the_import_says_so(monkeypatch):
    monkeypatch.setattr(hip, "_torch", None)
    monkeypatch.setitem(sys.modules, "torch", None)
    with pytest.raises(ImportError):
        HipBackend._stream()
