"""Calls without an explicit stream go to the caller's current stream."""
import pytest

from nerve_amd import hip

pytestmark = pytest.mark.gpu


def test_current_stream_handle(ctx, dev):
    import torch

    side = torch.cuda.Stream(dev)
    assert hip._stream(None) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert hip._stream(None) == side.cuda_stream == torch.cuda.current_stream().cuda_stream
        logits = torch.zeros(1, 64, dtype=torch.float32, device=dev)
        logits[0, 7] = 1.0
        out = torch.zeros(1, dtype=torch.int32, device=dev)
        ctx.argmax_f32(logits, 1, 64, out)
        side.synchronize()
        assert out.item() == 7
    assert hip._stream(side) == side.cuda_stream
