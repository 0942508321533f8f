"""The C calls' stream handle, GPU: torch's current stream, inside a stream context and outside, the raw handle where torch
offers it and the public one."""

import pytest
import torch

from blochparty_amd.engines import hip


@pytest.mark.gpu
@pytest.mark.parametrize("handle", [hip.raw_stream, hip._public_stream])
def test_handle_of_the_current_stream(gpu, handle):
    side, dev = torch.cuda.Stream(), torch.cuda.current_device()
    assert handle(dev) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert handle(dev) == side.cuda_stream != torch.cuda.default_stream().cuda_stream
