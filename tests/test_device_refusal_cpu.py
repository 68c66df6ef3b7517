"""Host tensors are refused before their addresses reach a kernel: the backward by itself (the forward
checks its inputs first), which is what a caller with saved tensors on the CPU reaches."""
import pytest
import torch

from gvv_amd import _lib, renderer


@pytest.fixture
def no_library(monkeypatch):
    class Library:
        def gvv_backward(self, *args):
            raise AssertionError("host addresses were passed to the library")

    monkeypatch.setattr(_lib, "load", lambda: Library())
    # a host with a device, whose current stream is the default one
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 0, raising=False)
    monkeypatch.setattr(renderer, "_raw_stream", lambda index: 0, raising=False)


def test_backward_refuses_host_tensors(no_library):
    r = renderer.Rasterizer.__new__(renderer.Rasterizer)
    r._h, r.N, r.C, r.W, r.H = None, 3, 1, 4, 4
    z = torch.zeros
    with pytest.raises(ValueError, match="cpu"):
        r.backward(z(1, 1, 4, 4, 3), None, None, z(1, 3, 3), z(1, 3, 3), z(1, 2, 2, 3), z(1, 1, 27), z(1, 1, 3, 3),
                   z((1, 1, 4, 4), dtype=torch.int32), z(1, 12), z(1, 9))


@pytest.mark.parametrize("device", ["cpu", "meta"])
def test_stream_of_another_device_is_refused(no_library, device):
    with pytest.raises(ValueError, match=device):
        renderer._stream_ptr(torch.device(device))


def test_stream_of_a_device(no_library, monkeypatch):
    monkeypatch.setattr(renderer, "_raw_stream", lambda index: 100 + index)
    assert renderer._stream_ptr(torch.device("cuda")) == 100
    assert renderer._stream_ptr(torch.device("cuda", 3)) == 103
