"""The C calls' stream handle, GPU: torch's current stream, inside a stream context and outside, also where torch does not
offer the raw handle."""

import pytest
import torch

from blochparty_amd.engines import hip


@pytest.mark.gpu
@pytest.mark.parametrize("offered", [True, False])
def test_handle_of_the_current_stream(gpu, monkeypatch, offered):
    if not offered:
        monkeypatch.setattr(hip, "_RAW_STREAM", None)
    side = torch.cuda.Stream()
    assert hip.raw_stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert hip.raw_stream() == side.cuda_stream != torch.cuda.default_stream().cuda_stream
