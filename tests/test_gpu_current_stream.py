"""Calls without a stream argument run on torch's current stream: the default one, a side stream
inside a stream context, and per thread."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_default_stream_argument_follows_torch(gpu):
    from holoflow_amd import hfx

    def handle():
        return hfx._stream(None).value or 0

    assert handle() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    seen = {}
    with torch.cuda.stream(side):
        assert handle() == side.cuda_stream
        x = torch.arange(1 << 16, device="cuda", dtype=torch.int32).to(torch.int16)
        y = hfx.convert_u16(x)
        t = threading.Thread(target=lambda: seen.update(h=handle()))
        t.start()
        t.join()
    side.synchronize()
    assert torch.equal(y.cpu(), (x.cpu().to(torch.int32) & 0xFFFF).float())
    assert seen["h"] == torch.cuda.default_stream().cuda_stream
    assert handle() == torch.cuda.current_stream().cuda_stream
