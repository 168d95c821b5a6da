"""The stream handle that device calls take when none is given is torch's
current stream, on the default stream and inside a stream context."""
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
