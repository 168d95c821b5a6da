"""The stream handle that device calls take when none is given is torch's
current stream, on the default stream and inside a stream context, and with a
torch that lacks the private functions it is read with."""
import pytest

from drifter_amd import solver


@pytest.mark.gpu
def test_handle_is_the_current_stream():
    import torch

    torch.zeros(1, device="cuda")
    assert (solver._sptr(None).value or 0) == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert solver._sptr(None).value == side.cuda_stream
    assert solver._sptr(side).value == side.cuda_stream
    assert (solver._sptr(None).value or 0) == torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("missing", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_handle_without_torchs_private_functions(monkeypatch, missing):
    """A torch build that lacks them gives the handle of its Stream object."""
    import types

    import torch

    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda: types.SimpleNamespace(cuda_stream=1234))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: 5678, raising=False)
    assert solver._sptr(None).value == 5678
    monkeypatch.delattr(torch._C, missing)
    assert solver._sptr(None).value == 1234
