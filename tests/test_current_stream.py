"""A launch without a stream goes to torch's current stream of the current
device, inside and outside a stream context."""
import pytest


@pytest.mark.gpu
def test_launches_follow_the_current_stream(fa_lib):
    import torch

    assert fa_lib._stream(None) == torch.cuda.current_stream().cuda_stream
    for side in (torch.cuda.Stream(), torch.cuda.Stream()):
        with torch.cuda.stream(side):
            assert fa_lib._stream(None) == side.cuda_stream != 0
    assert fa_lib._stream(None) == torch.cuda.current_stream().cuda_stream
    assert fa_lib._stream(side) == side.cuda_stream and fa_lib._stream(0) == 0
